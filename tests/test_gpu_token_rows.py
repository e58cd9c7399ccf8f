"""GPU: Q read and O written in token order with tiled K and V (li_bsa_fwd_qo) against the tile / attend / untile
sequence, bit for bit: 64- and 128-token tiles, both head dims and element types, e4m3, odd grids, split tiles, ragged
rows longest first, and the query views that still need Q tiles."""
import math

import pytest
import torch

from li_sparse import _core, _pipeline
from li_sparse.hy.ar_sparse_operation import fast_generate_indices

pytestmark = pytest.mark.gpu

CASES = [  # B, H, D, dtype, tile, (H, W), frames q / k, text, e4m3, row budgets, layout
    (1, 3, 64, torch.bfloat16, (4, 4, 4), (11, 14), 5, 6, 33, False, False, "blhd"),
    (2, 2, 64, torch.float16, (4, 4, 4), (8, 8), 4, 4, 0, False, False, "bhld"),
    (1, 2, 64, torch.bfloat16, (4, 8, 4), (9, 30), 1, 4, 0, False, False, "blhd"),
    (1, 2, 128, torch.float16, (4, 4, 4), (10, 9), 3, 8, 70, False, False, "bhld"),
    (2, 3, 128, torch.bfloat16, (2, 8, 8), (13, 21), 3, 7, 200, False, False, "blhd"),
    (1, 4, 128, torch.float16, (4, 8, 4), (17, 30), 4, 8, 1, False, True, "blhd"),
    (1, 3, 128, torch.bfloat16, (4, 4, 8), (22, 41), 4, 8, 130, True, False, "blhd"),
    (1, 16, 128, torch.bfloat16, (4, 8, 4), (30, 53), 4, 4, 0, False, False, "bhld"),
]


def _bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("case", CASES)
def test_equals_tile_attend_untile(dev, case):
    B, NH, D, dtype, tile, hw, fq, fk, text, fp8, ragged, layout = case
    print(f"[gpu] token-order Q / O, tiled K / V: {case}", flush=True)
    gen, tok = torch.Generator().manual_seed(11), hw[0] * hw[1]

    def make(L):
        x = torch.randn(B, L, NH, D, generator=gen).to(dtype).to(dev).permute(0, 2, 1, 3)
        return x if layout == "blhd" else x.contiguous()

    q, k, v, kt, vt = make(fq * tok), make(fk * tok), make(fk * tok), make(text), make(text)
    g = _pipeline.geometry(hw, tile, fq * tok, fk * tok, text)
    params = {"tile_size": tile, "topk_ratio": 0.4, "sim_metric": "scaled_dot_product", "force_diag": True}
    if ragged:
        params["row_budget"] = [2 + (7 * i) % g.nk_blk for i in range(g.nq_blk)]

    def select(qp, kp, tl, gq, gk):
        return fast_generate_indices(qp, kp, tl, gq, gk, params, dev)

    txt = (kt, vt) if text else (None, None)
    run = lambda x: _pipeline.sparse_attention(x, *txt, k, v, hw, tile, select, fused=False,  # noqa: E731
                                               balance=ragged, qk_fp8=fp8)
    got = run(q)
    # a view whose rows cannot be read 16 bytes at a time takes Q tiles and the untile pass
    odd = torch.stack([q, q], -1)[..., 0]
    assert not _pipeline._token_rows(odd)
    other = run(odd)
    # the sequence itself
    geo_q, geo_k = (g.T_q, *hw, *tile, g.nh, g.nw), (g.T_k, *hw, *tile, g.nh, g.nw)
    code = _core.FP8 if fp8 else dtype
    q_t, k_t = (torch.empty((B, NH, n, g.bs, D), dtype=code, device=dev) for n in
                (g.nq_blk, g.num_txt_blk + g.nk_blk))
    v_t = torch.empty(k_t.shape, dtype=dtype, device=dev)
    q_s, k_s = (torch.empty((B, NH, x.shape[2]), device=dev) if fp8 else None for x in (q_t, k_t))
    qp, kp = (torch.empty((B, NH, n, D), dtype=dtype, device=dev) for n in (g.nq_blk, g.nk_blk))
    _core.prep(q, qp, geo_q, k, v, kp, 0, geo_k, q_tiles=q_t, q_scale=q_s, k_tiles=k_t, k_scale=k_s, v_tiles=v_t,
               num_txt_blk=g.num_txt_blk, text=(kt, vt) if text else None)
    ind, cnt = select(qp, kp, text, (g.nt_q, g.nh, g.nw), (g.nt_k, g.nh, g.nw))
    flat, scale = lambda x: x.flatten(2, 3), 1.0 / math.sqrt(D)  # noqa: E731
    if fp8:
        o, lse = _core.bsa_forward_fp8(flat(q_t), q_s, flat(k_t), k_s, flat(v_t), ind, cnt, scale, g.bs,
                                       return_lse=True, balance=ragged)
    else:
        o, lse = _core.bsa_forward(flat(q_t), flat(k_t), flat(v_t), ind, cnt, scale, g.bs, return_lse=True,
                                   balance=ragged)
    ref = torch.empty_like(q)
    _core.untile(o.view(B, NH, g.nq_blk, g.bs, D), ref, *geo_q)
    out, lse2 = _core.bsa_forward_qo(q_t if fp8 else q, k_t, v_t, geo_q, ind, cnt, scale, torch.empty_like(q),
                                     q_scale=q_s, k_scale=k_s, return_lse=True, balance=ragged)
    torch.cuda.synchronize()
    assert got.stride() == q.stride()
    for x in (got, other, out):
        assert torch.equal(_bits(x), _bits(ref))
    assert torch.equal(lse.view(torch.int32), lse2.view(torch.int32))


def test_rejects_what_the_kernel_does_not_take(dev):
    q = torch.zeros(1, 2, 128, 64, dtype=torch.bfloat16, device=dev)
    kt = torch.zeros(1, 2, 3, 64, 64, dtype=torch.bfloat16, device=dev)
    ind, cnt = torch.zeros(1, 2, 2, 1, dtype=torch.int32, device=dev), torch.ones(1, 2, 2, dtype=torch.int32, device=dev)
    geo = (2, 8, 8, 1, 8, 8, 1, 1)
    call = lambda q=q, k=kt, v=kt, geo=geo, ind=ind, out=q: _core.bsa_forward_qo(  # noqa: E731
        q, k, v, geo, ind, cnt, 0.1, torch.empty_like(out))
    call()
    for kw in (dict(q=q[:, :, :100]), dict(v=kt[:, :, :2].contiguous()), dict(k=kt[:, :, ::2], v=kt[:, :, ::2]),
               dict(geo=(2, 8, 8, 1, 4, 8, 2, 1)), dict(geo=(2, 8, 8, 1, 8, 8, 2, 1)), dict(ind=ind[:, :, :1]),
               dict(out=torch.zeros(1, 2, 100, 64, dtype=torch.bfloat16, device=dev)),
               dict(q=torch.stack([q, q], -1)[..., 0])):
        with pytest.raises(RuntimeError):
            call(**kw)


# one tile per CU at most (four interleaves for lists of more than ten blocks, else two), more (two)
@pytest.mark.parametrize("H,nq", [(2, 3), (8, 40)])
@pytest.mark.parametrize("cols", [1, 4, 5, 10, 11, 13])
def test_64_dim_kernel_against_float64(dev, H, nq, cols):
    """Lists around the interleaves' counts, empty lists, ids out of range, a partial last tile: 2e-2 as elsewhere (P and
    the output in bf16), LSE 1e-3."""
    import numpy as np
    from helpers import bits
    from oracle import attention as oatt
    from oracle.bf16 import bf16_to_f32

    print(f"[gpu] 64-dim kernel H={H} nq={nq} cols={cols}", flush=True)
    bs, D, nkb = 64, 64, 15
    Lq = nq * bs - 23
    gen = torch.Generator().manual_seed(cols)
    q, k, v = (torch.randn(1, H, n, D, generator=gen).to(torch.bfloat16) for n in (Lq, nkb * bs, nkb * bs))
    rng = np.random.default_rng(cols)
    ind = np.argsort(rng.random((1, H, nq, nkb)), axis=-1)[..., :cols].astype(np.int32)
    cnt = rng.integers(0, cols + 1, size=(1, H, nq)).astype(np.int32)
    bad = ind.copy()
    bad[0, 0, :, 0] = [nkb, -1, 2 ** 30][cols % 3]   # the kernel adds nothing for these
    o, lse = _core.bsa_forward(q.to(dev), k.to(dev), v.to(dev), torch.from_numpy(bad).to(dev),
                               torch.from_numpy(cnt).to(dev), 0.125, bs, return_lse=True)
    torch.cuda.synchronize()
    good, n = ind.copy(), cnt.copy()
    for m in range(nq):
        if n[0, 0, m] > 0:
            good[0, 0, m, :-1], n[0, 0, m] = ind[0, 0, m, 1:], n[0, 0, m] - 1
    f64 = lambda t: bf16_to_f32(bits(t)).astype(np.float64)  # noqa: E731
    o_ref, lse_ref = oatt.bsa_forward(f64(q), f64(k), f64(v), good, n, 0.125, bs)
    got, fin = lse.cpu().numpy(), np.isfinite(lse_ref)
    assert np.array_equal(np.isneginf(got), ~fin)
    assert np.abs(o.float().cpu().numpy() - o_ref).max() <= 2e-2
    assert not fin.any() or np.abs(got[fin] - lse_ref[fin]).max() <= 1e-3


@pytest.mark.parametrize("H,nq", [(2, 3), (8, 40)])
def test_64_dim_kernel_keeps_nan(dev, H, nq):
    """A query row with a NaN (every score NaN) has NaN outputs and a NaN LSE; an empty list zeros and -inf."""
    print(f"[gpu] 64-dim kernel, NaN rows H={H} nq={nq}", flush=True)
    bs, D, nkb = 64, 64, 12
    gen = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(1, H, n * bs, D, generator=gen).to(torch.bfloat16).to(dev) for n in (nq, nkb, nkb))
    q[0, 0, 5, 7] = q[0, 1, bs + 60] = float("nan")
    ind = torch.arange(nkb, dtype=torch.int32, device=dev).repeat(1, H, nq, 1)
    cnt = torch.full((1, H, nq), nkb, dtype=torch.int32, device=dev)
    cnt[0, 0, 1] = 0
    o, lse = _core.bsa_forward(q, k, v, ind, cnt, 0.125, bs, return_lse=True)
    torch.cuda.synchronize()
    want = torch.zeros(1, H, nq * bs, dtype=torch.bool, device=dev)
    want[0, 0, 5] = want[0, 1, bs + 60] = True
    assert torch.equal(torch.isnan(o).all(-1), want) and torch.equal(torch.isnan(o).any(-1), want)
    assert torch.equal(torch.isnan(lse), want)
    assert torch.isneginf(lse[0, 0, bs:2 * bs]).all() and not o[0, 0, bs:2 * bs].any()

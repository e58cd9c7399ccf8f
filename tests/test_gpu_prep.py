"""GPU: the one-launch preparation (li_prep) against the single gathers and pools, bit for bit.

Odd grids and text lengths, vector and element-wise strides (also mixed in one call), both head dims and element types.
"""
import pytest
import torch

from li_sparse import _core
from li_sparse._ops import ops

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.uint8 if t.element_size() == 1 else torch.int16 if t.element_size() == 2 else torch.int32)


def _tok(gen, B, H, L, D, dtype, dev, how):
    x = torch.randn(B, L, H, D, generator=gen).to(dtype).to(dev)
    if how == "blhd":
        return x.permute(0, 2, 1, 3)
    if how == "dstride2":     # element-wise: d stride 2
        return torch.stack([x, x], -1).permute(0, 2, 1, 3, 4)[..., 0]
    return x.permute(0, 2, 1, 3).contiguous()


CASES = [  # D, dtype, tile, (H, W), frames q / k, first key frame, text, layouts of q, k, v, text
    (128, torch.bfloat16, (4, 8, 4), (17, 30), 3, 6, 0, 77, "bhld", "bhld", "blhd", "bhld"),
    (128, torch.float16, (2, 8, 8), (9, 13), 1, 4, 2, 0, "blhd", "blhd", "blhd", "bhld"),
    (128, torch.bfloat16, (4, 4, 8), (5, 24), 4, 4, 4, 128, "blhd", "blhd", "blhd", "blhd"),   # no key block left
    (128, torch.bfloat16, (2, 8, 8), (16, 16), 2, 3, 0, 129, "dstride2", "blhd", "bhld", "dstride2"),
    (64, torch.bfloat16, (4, 4, 4), (11, 7), 5, 5, 0, 1, "bhld", "dstride2", "dstride2", "bhld"),
    (64, torch.float16, (4, 4, 4), (8, 8), 4, 8, 4, 64, "blhd", "blhd", "bhld", "blhd"),
]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("case", CASES)
def test_prep_equals_single_launches(dev, case, fp8):
    D, dtype, tile, (H, W), fq, fk, first, text, lq, lk, lv, lt = case
    print(f"[gpu] prep {case} fp8={fp8}", flush=True)
    gen = torch.Generator().manual_seed(5)
    B, NH = 2, 3
    tt, th, tw = tile
    bs, nh, nw = tt * th * tw, -(-H // th), -(-W // tw)
    q, k, v = (_tok(gen, B, NH, f * H * W, D, dtype, dev, l) for f, l in ((fq, lq), (fk, lk), (fk, lv)))
    kt, vt = (_tok(gen, B, NH, text, D, dtype, dev, lt) for _ in range(2))
    ntxt, fb = -(-text // bs), first // tt * nh * nw
    nq, nk = -(-fq // tt) * nh * nw, -(-fk // tt) * nh * nw
    gq, gk = (fq, H, W, tt, th, tw, nh, nw), (fk - first, H, W, tt, th, tw, nh, nw)
    kv, vv = k[:, :, first * H * W:], v[:, :, first * H * W:]

    def buffers():
        code = torch.float8_e4m3fn if fp8 else dtype
        fill = lambda shape, dt: torch.full(shape, 1.0, dtype=dt, device=dev)  # noqa: E731
        return dict(q_tiles=fill((B, NH, nq, bs, D), code), q_scale=fill((B, NH, nq), torch.float32) if fp8 else None,
                    k_tiles=fill((B, NH, ntxt + nk, bs, D), code),
                    k_scale=fill((B, NH, ntxt + nk), torch.float32) if fp8 else None,
                    v_tiles=fill((B, NH, ntxt + nk, bs, D), dtype), q_pool=fill((B, NH, nq, D), dtype),
                    k_pool=fill((B, NH, nk, D), dtype))

    a, b = buffers(), buffers()
    k_n = torch.ones_like(a["k_pool"])
    _core.prep(q, a["q_pool"], gq, kv, vv, a["k_pool"], fb, gk, q_tiles=a["q_tiles"], q_scale=a["q_scale"],
               k_tiles=a["k_tiles"], k_scale=a["k_scale"], v_tiles=a["v_tiles"], k_pool_n=k_n, num_txt_blk=ntxt,
               text=(kt, vt) if text else None)
    pad = (0, 0, 0, ntxt * bs - text)
    kp, vp = (torch.nn.functional.pad(x, pad).contiguous() for x in (kt, vt))
    if fp8:
        _core.tile_prep_fp8(q, b["q_tiles"], b["q_scale"], b["q_pool"], 0, 0, *gq)
        if first < fk:
            _core.kv_prep_fp8(kv, vv, b["k_tiles"], b["k_scale"], b["v_tiles"], b["k_pool"], ntxt + fb, fb, *gk)
        if text:
            _core.tile_prep_fp8(kp, b["k_tiles"], b["k_scale"], None, 0, 0, ntxt, 1, bs, 1, 1, bs, 1, 1)
    else:
        _core.q_prep(q, b["q_tiles"], b["q_pool"], *gq)
        if first < fk:
            _core.kv_prep(kv, vv, b["k_tiles"], b["v_tiles"], b["k_pool"], ntxt + fb, fb, *gk)
        if text:
            b["k_tiles"][:, :, :ntxt].copy_(kp.view(B, NH, ntxt, bs, D))
    if text:
        b["v_tiles"][:, :, :ntxt].copy_(vp.view(B, NH, ntxt, bs, D))
    torch.cuda.synchronize()
    for name, x in a.items():
        assert x is None or torch.equal(_bits(x), _bits(b[name])), name
    if first < fk:
        qp, ref, ref_n = torch.empty_like(a["q_pool"]), torch.ones_like(k_n), torch.ones_like(k_n)
        _core.pool_pair(q, qp, 0, gq, kv, ref, fb, gk, mean1_normalized=ref_n)
        torch.cuda.synchronize()
        assert torch.equal(_bits(qp), _bits(a["q_pool"])) and torch.equal(_bits(ref), _bits(a["k_pool"]))
        assert torch.equal(_bits(ref_n), _bits(k_n))
    if text:   # padded rows instead of leading tiles, and on their own
        rows = [torch.ones_like(kp), torch.ones_like(vp)]
        _core.prep(q, a["q_pool"], gq, kv, vv, a["k_pool"], fb, gk, num_txt_blk=ntxt, text=(kt, vt), padded_text=rows)
        alone = _core.pad_text(kt, vt, bs)
        torch.cuda.synchronize()
        for got in (rows, alone):
            assert torch.equal(_bits(got[0]), _bits(kp)) and torch.equal(_bits(got[1]), _bits(vp))


def test_prep_rejects_short_tensors(dev):
    q = torch.zeros(1, 2, 2 * 64, 128, dtype=torch.bfloat16, device=dev)
    pool = torch.zeros(1, 2, 1, 128, dtype=torch.bfloat16, device=dev)
    g = [2, 8, 8, 2, 8, 8, 1, 1]
    txt = torch.zeros(1, 2, 100, 128, dtype=torch.bfloat16, device=dev)
    short = torch.zeros(1, 2, 100, 128, dtype=torch.bfloat16, device=dev)
    call = lambda **kw: ops.prep(*[dict(q=q, q_tiles=None, q_scale=None, q_pool=pool, q_geom=g, k=q, v=q,  # noqa: E731
                                        k_tiles=None, k_scale=None, v_tiles=None, k_pool=pool, k_pool_n=None, first=0,
                                        k_geom=g, num_txt_blk=1, k_txt=txt, v_txt=txt, txt_k=None, txt_v=None,
                                        **{})[n] if n not in kw else kw[n] for n in
                                   ("q", "q_tiles", "q_scale", "q_pool", "q_geom", "k", "v", "k_tiles", "k_scale",
                                    "v_tiles", "k_pool", "k_pool_n", "first", "k_geom", "num_txt_blk", "k_txt", "v_txt",
                                    "txt_k", "txt_v")])
    call()
    for bad in (dict(txt_k=short), dict(num_txt_blk=2), dict(k=q[:, :, :100]), dict(first=1), dict(v_txt=None),
                dict(q_tiles=short), dict(k_pool_n=pool[:, :1])):
        with pytest.raises(RuntimeError):
            call(**bad)


@pytest.mark.parametrize("text", [77, 128])
def test_text_of_another_type_or_device(dev, text):
    """K / V tiles take text as a copy into them would; e4m3 codes are those of the 16-bit text keys as they came;
    what reads the text in place, or quantizes 32-bit keys, refuses it."""
    from li_sparse import ContextCache, _pipeline
    from li_sparse.hy.ar_sparse_operation import fast_generate_indices

    print(f"[gpu] text of another type: {text} tokens", flush=True)
    gen, tile, NH, D = torch.Generator().manual_seed(9), (4, 8, 4), 2, 128
    params = {"tile_size": tile, "topk_ratio": 0.5, "sim_metric": "scaled_dot_product"}
    kt, vt = (torch.randn(1, NH, text, D, generator=gen).to(dev) for _ in range(2))

    def call(hw, kt, vt, fp8, cache=None):
        q, k = (_tok(torch.Generator().manual_seed(f), 1, NH, f * hw[0] * hw[1], D, torch.bfloat16, dev, "bhld")
                for f in (3, 5))
        return _pipeline.sparse_attention(
            q, kt, vt, k, k, hw, tile, lambda qp, kp, tl, gq, gk: fast_generate_indices(qp, kp, tl, gq, gk, params, dev),
            qk_fp8=fp8, context=(cache, 0, 4) if cache is not None else None)

    odd, even = (9, 13), (9, 16)       # K / V tiles; tokens read in place
    ref = call(odd, kt.bfloat16(), vt.bfloat16(), False)
    for a, b in ((kt, vt), (kt.cpu(), vt.cpu()), (kt.bfloat16(), vt.cpu())):
        assert torch.equal(_bits(call(odd, a, b, False)), _bits(ref))
    cache, n = ContextCache(), -(-text // 128)
    half = kt.half()
    out = call(odd, half, vt, True, cache)
    bufs = next(iter(cache._entries.values()))
    codes = torch.empty((1, NH, n, 128, D), dtype=torch.float8_e4m3fn, device=dev)
    scales = torch.empty((1, NH, n), device=dev)
    rows = torch.nn.functional.pad(half, (0, 0, 0, n * 128 - text))
    _core.tile_prep_fp8(rows, codes, scales, None, 0, 0, n, 1, 128, 1, 1, 128, 1, 1)
    assert torch.equal(_bits(bufs["k8"][:, :, :n].contiguous()), _bits(codes))
    assert torch.equal(_bits(bufs["k_scale"][:, :, :n].contiguous()), _bits(scales))
    assert torch.equal(_bits(call(odd, half, vt, True, cache)), _bits(out))   # the second call keeps them
    for hw, a, b, fp8 in ((odd, kt, vt, True), (even, kt, vt.bfloat16(), True), (even, half, half, True),
                          (even, kt.bfloat16(), vt, False), (even, half, half, False)):
        with pytest.raises((TypeError, RuntimeError)):
            call(hw, a, b, fp8)
    torch.cuda.synchronize()

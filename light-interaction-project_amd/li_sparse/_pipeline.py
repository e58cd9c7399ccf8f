"""The sparse-attention call shared by the HY and MG entry points.

Steps (ar_sparse_operation.py:316-362, bi_sparse_operation_for_KV_cache.py:347-395,
bi_sparse_operation.py:246-348): block geometry; one launch that pools Q and K,
zero-pads text K/V into the leading blocks and, where the attention kernel
cannot read the tokens in place, gathers tiles; block selection; block-sparse
attention into ``empty_like(q)``.  The index lists come from the mask kernel, so
the attention launch needs no host-side range check (the reference's ``block_indices.max()`` sync is gone).
"""
import math
from dataclasses import dataclass
from numbers import Real
from operator import index

import numpy as np
import torch
import torch.nn.functional as F

from . import _core, _lib
from ._ops import ops

_sparse_call = ops.sparse_call.default


@dataclass(frozen=True)
class Geometry:
    """Block geometry of one call (ar_sparse_operation.py:319-327)."""
    H: int
    W: int
    tt: int
    th: int
    tw: int
    bs: int
    nh: int
    nw: int
    T_q: int
    T_k: int
    nt_q: int
    nt_k: int
    num_txt_blk: int
    nq_blk: int
    nk_blk: int


def pad_blocks(x, t):
    return (x + (t - x % t) % t) // t


def geometry(latent_hw, tile, vis_len_q, vis_len_k, text_len):
    H, W = latent_hw
    tt, th, tw = tile
    bs = tt * th * tw
    nh, nw = pad_blocks(H, th), pad_blocks(W, tw)
    T_q, T_k = vis_len_q // (H * W), vis_len_k // (H * W)
    nt_q, nt_k = pad_blocks(T_q, tt), pad_blocks(T_k, tt)
    num_txt_blk = pad_blocks(text_len, bs)
    return Geometry(H, W, tt, th, tw, bs, nh, nw, T_q, T_k, nt_q, nt_k, num_txt_blk, nt_q * nh * nw, nt_k * nh * nw)


def _stage(events, name):
    if events is not None:
        e = torch.cuda.Event(enable_timing=True)
        e.record()
        events[name] = e


def _fusable(*ts):
    """Token views the fused kernel reads directly: unit d stride, 16-byte aligned, non-overlapping rows."""
    for t in ts:
        st = t.stride()
        if st[3] != 1 or any(x % 8 for x in st[:3]) or st[2] < t.shape[3] or t.data_ptr() % 16:
            return False
    return True


def _token_rows(*ts):
    """Token views whose rows the tiled-K/V kernels read (Q) and write (O): unit d stride, 16-byte aligned rows."""
    for t in ts:
        st = t.stride()
        if st[3] != 1 or any(x % 8 for x in st[:3]) or st[2] <= 0 or t.data_ptr() % 16:
            return False
    return True


def uses_fused(q, k_vis, v_vis, tile, latent_hw):
    """True when ``sparse_attention(..., fused=True)`` takes the fused kernel for these inputs."""
    return _core.fused_supported(q.shape[3], tile, latent_hw) and _fusable(q, k_vis, v_vis)


def ragged(sparse_params):
    """Whether the rows have their own budgets (then the attention starts its longest tiles first)."""
    return sparse_params.get("row_budget") is not None


def qk_fp8(sparse_params):
    """The ``qk_fp8`` extension key: Q K^T on e4m3 codes with per-tile-block scales."""
    return bool(sparse_params.get("qk_fp8", False))


def cosine(sparse_params):
    """Whether the selection scores blocks by cosine similarity (the reference's default ``sim_metric``)."""
    return sparse_params.get("sim_metric", "cosine") == "cosine"


class ContextCache:
    """Prepared key-side blocks of the fixed context of K/V, kept across calls.

    HY-WorldPlay recomputes the current chunk's K/V at every denoise step while
    the memory frames' K/V and the text stay fixed for the chunk; the reference
    re-tiles all of it on every call (ar_sparse_operation.py:337-348).  Pass a
    cache as ``sparse_params["context_cache"]`` with
    ``sparse_params["context_frames"]``, the number of leading K frames that do
    not change until the next ``reset()``.  The first call per layer
    (``block_idx``) and shape prepares every key block (pools; e4m3 codes and
    scales; tiles on the tiled paths) and keeps the buffers; later calls
    prepare only the blocks from the first t-slab that is not entirely
    context (the context is rounded down to whole ``tt``-frame slabs) and the
    text blocks not at all.  Results are bit-identical to uncached calls.  Call
    ``reset()`` whenever the context or the text changes (a new chunk);
    calls that share a cache must run on one stream.
    """

    def __init__(self):
        self._entries = {}

    def reset(self):
        self._entries.clear()

    def __len__(self):
        return len(self._entries)


def context_of(sparse_params, block_idx):
    """(cache, layer, frames) from ``sparse_params`` for ``sparse_attention``, or None without a cache."""
    cache = sparse_params.get("context_cache")
    if cache is None:
        return None
    if not isinstance(cache, ContextCache):
        raise TypeError("sparse_params['context_cache'] must be a li_sparse.ContextCache")
    return cache, block_idx, int(sparse_params.get("context_frames", 0))


def _prepare(path, q, k_txt, v_txt, k_vis, v_vis, g, text_len, ctx, k_norm):
    """What one call prepares of its tensors, in one launch (li_prep): a dict of the buffers.

    path: "fused" (pools; padded text K/V), "fused_fp8" (e4m3 Q and K tiles + scales, pools; padded text V), "mixed"
    (K, V tiles, pools), "tiled" (Q, K, V tiles, pools), "mixed_fp8" and "tiled_fp8" (e4m3 Q and K tiles + scales, V
    tiles, pools).  Query-side buffers are the call's own; key-side ones (text blocks, then the visual blocks from the
    first uncached frame) are the ContextCache's where there is one.  k_norm: also keep the K pool's rows normalised for
    the cosine selection (``k_pool_n``; the selection takes it as ``k_pool_normalized``).
    """
    B, NH, _, D = q.shape
    dt = q.dtype
    fp8, tiled = path.endswith("_fp8"), not path.startswith("fused")
    cache, layer, cframes = ctx if ctx is not None else (None, None, 0)
    cf = min((max(cframes, 0) // g.tt) * g.tt, g.T_k) if cache is not None else 0
    key = (path, layer, B, NH, D, dt, str(q.device), g, text_len, cf, bool(k_norm)) if cache is not None else None
    bufs = cache._entries.get(key) if cache is not None else None
    first = cf if bufs is not None else 0
    text, padded, k_codes = None, (None, None), None
    if bufs is None:
        nkb = g.num_txt_blk + g.nk_blk
        bufs = dict.fromkeys(("k_pool_n", "k8", "k_scale", "k_all", "v_all", "kt", "vt"))
        bufs["k_pool"] = q.new_empty((B, NH, g.nk_blk, D))
        if k_norm:
            bufs["k_pool_n"] = torch.empty_like(bufs["k_pool"])
        if fp8:
            bufs["k8"] = q.new_empty((B, NH, nkb, g.bs, D), dtype=_core.FP8)
            bufs["k_scale"] = q.new_empty((B, NH, nkb), dtype=torch.float32)
        elif tiled:
            bufs["k_all"] = q.new_empty((B, NH, nkb, g.bs, D))
        if tiled:
            bufs["v_all"] = q.new_empty((B, NH, nkb, g.bs, D))
        if text_len > 0:
            if tiled:
                # Tiles take text of another element type (16-bit ones of another device too) as a copy into them
                # would; e4m3 codes are those of the 16-bit keys as they came.
                if fp8:
                    _core._device_check(q, k_txt)
                    _core.dtype_code(k_txt)
                    k_codes = k_txt if k_txt.dtype != dt else None
                k_txt, v_txt = k_txt.to(q), v_txt.to(q)
            else:
                _core._same_dtype(q, k_txt, v_txt)
            text = (k_txt, v_txt)
            # Whole blocks of text are read where they are.
            whole = text_len % g.bs == 0
            if path == "fused":
                bufs["kt"], keep_k = _text_rows(k_txt, g, whole)
                padded = (None if keep_k else bufs["kt"], None)
            if not tiled:
                bufs["vt"], keep_v = _text_rows(v_txt, g, whole)
                padded = (padded[0], None if keep_v else bufs["vt"])
    out = dict(bufs, q_pool=q.new_empty((B, NH, g.nq_blk, D)), q_tiles=None, q_scale=None)
    if fp8:
        out["q_tiles"] = q.new_empty((B, NH, g.nq_blk, g.bs, D), dtype=_core.FP8)
        out["q_scale"] = q.new_empty((B, NH, g.nq_blk), dtype=torch.float32)
    elif path == "tiled":
        out["q_tiles"] = q.new_empty((B, NH, g.nq_blk, g.bs, D))
    if first > 0:
        k_vis, v_vis = k_vis[:, :, first * g.H * g.W:], v_vis[:, :, first * g.H * g.W:]
    rest = (g.H, g.W, g.tt, g.th, g.tw, g.nh, g.nw)
    _core.prep(q, out["q_pool"], (g.T_q, *rest), k_vis, v_vis, bufs["k_pool"], (first // g.tt) * g.nh * g.nw,
               (g.T_k - first, *rest), q_tiles=out["q_tiles"], q_scale=out["q_scale"],
               k_tiles=bufs["k8"] if fp8 else bufs["k_all"], k_scale=bufs["k_scale"], v_tiles=bufs["v_all"],
               k_pool_n=bufs["k_pool_n"], num_txt_blk=g.num_txt_blk, text=text, padded_text=padded)
    if k_codes is not None:
        _core.tile_prep_fp8(k_codes, bufs["k8"], bufs["k_scale"], None, 0, 0, 1, 1, text_len, 1, 1, g.bs, 1, g.num_txt_blk)
    if cache is not None:
        cache._entries[key] = bufs
    return out


def _text_rows(x, g, whole):
    """(padded text buffer, True if it is ``x`` itself)."""
    if whole and x.is_contiguous():
        return x, True
    return x.new_empty((*x.shape[:2], g.num_txt_blk * g.bs, x.shape[3])), False


def _select(select, kb, text_len, g):
    """``select`` on the call's pools; the normalised key pool goes along only when the call wrote one."""
    kw = {} if kb["k_pool_n"] is None else {"k_pool_normalized": kb["k_pool_n"]}
    return select(kb["q_pool"], kb["k_pool"], text_len, (g.nt_q, g.nh, g.nw), (g.nt_k, g.nh, g.nw), **kw)


def fp8_supported(D, tile):
    """Shapes the e4m3 (qk_fp8) path is built for: D = 128 and 128-token tiles."""
    return D == 128 and tile[0] * tile[1] * tile[2] == 128


def _call(path, q, k_txt, v_txt, k_vis, v_vis, o_out, g, select, text_len, events, balance, ctx, sorted_lists, k_norm):
    """Preparation, block selection, attention into ``o_out``, and the untile of the tiled paths."""
    B, NH, _, D = q.shape
    scale = 1.0 / math.sqrt(D)
    _stage(events, "prep_start")
    kb = _prepare(path, q, k_txt, v_txt, k_vis, v_vis, g, text_len, ctx, k_norm)
    _stage(events, "prep_end")
    _stage(events, "index_start")
    indices, counts = _select(select, kb, text_len, g)
    _stage(events, "index_end")
    _stage(events, "attn_start")
    grid = (g.num_txt_blk, g.T_q, g.T_k, g.H, g.W, g.tt, g.th, g.tw, g.nh, g.nw)
    o_flat = None
    if path == "fused":
        _core.bsa_forward_gather(q, k_vis, v_vis, kb["kt"], kb["vt"], *grid, indices, counts, scale, o_out,
                                 balance=balance, sorted_lists=sorted_lists)
    elif path == "fused_fp8":
        _core.bsa_forward_fp8_gather(kb["q_tiles"].flatten(2, 3), kb["q_scale"], kb["k8"].flatten(2, 3), kb["k_scale"],
                                     v_vis, kb["vt"], *grid, indices, counts, scale, o_out, balance=balance,
                                     sorted_lists=sorted_lists)
    elif path.startswith("mixed"):
        fp8 = path == "mixed_fp8"
        _core.bsa_forward_qo(kb["q_tiles"] if fp8 else q, kb["k8"] if fp8 else kb["k_all"], kb["v_all"],
                             (g.T_q, g.H, g.W, g.tt, g.th, g.tw, g.nh, g.nw), indices, counts, scale, o_out,
                             q_scale=kb["q_scale"], k_scale=kb["k_scale"], balance=balance)
    elif path == "tiled_fp8":
        o_flat = _core.bsa_forward_fp8(kb["q_tiles"].flatten(2, 3), kb["q_scale"], kb["k8"].flatten(2, 3),
                                       kb["k_scale"], kb["v_all"].flatten(2, 3), indices, counts, scale, g.bs,
                                       balance=balance)
    else:
        o_flat = _core.bsa_forward(kb["q_tiles"].flatten(2, 3), kb["k_all"].flatten(2, 3), kb["v_all"].flatten(2, 3),
                                   indices, counts, scale, g.bs, balance=balance)
    _stage(events, "attn_end")
    _stage(events, "untile_start")
    if o_flat is not None:
        _core.untile(o_flat.view(B, NH, g.nq_blk, g.bs, D), o_out, *grid[1:2], *grid[3:])
    _stage(events, "untile_end")


def sparse_attention(q, k_txt, v_txt, k_vis, v_vis, latent_hw, tile, select, events=None, fused=True,
                     balance=False, qk_fp8=False, context=None, normalize_k_pool=False, sorted_lists=False):
    """One sparse-attention forward.

    q (B,H,Lq,D); k_txt/v_txt (B,H,N_txt,D) or None; k_vis/v_vis (B,H,Lk,D), any strides.
    ``select(q_pool, k_pool, text_len, grid_q, grid_k) -> (indices, counts)``.  ``sorted_lists``: every
    row ``select`` returns lists its text blocks before its visual blocks, as the block mask's ascending
    lists do; the token-order kernels then take their faster load path (a text block listed after a
    visual block would read as zeros, so leave it off for other selectors).
    ``events`` (dict or None) collects CUDA events per stage for profiling.
    ``fused`` (default) runs pools + one gather/attend/untile kernel where the
    shape allows it (D = 128, 128-token tiles, tw and W multiples of 4, a grid
    at least one tile high and wide, token views with unit d stride);
    otherwise, or with ``fused=False``, K and V are tiled first and the kernel reads Q and writes O in
    token order (or Q is tiled and O untiled too, for views it cannot read).  All give the same bits.
    ``balance`` (rows with their own budgets) starts the longest query tiles first.  ``qk_fp8`` takes Q K^T on e4m3 codes with one scale per tile
    block (bf16 only; D = 128 and 128-token tiles, ValueError otherwise); the selection is unchanged.
    ``context`` = (ContextCache, layer key, context frames) keeps the key-side preparation of the
    fixed leading frames and the text across calls (see ContextCache).  ``normalize_k_pool`` (``select``
    scores by cosine similarity): the preparation also writes the key pool's rows
    normalised, once per key block, and the block mask takes them instead of normalising every key row in
    every workgroup of query rows (same selection, bit for bit); ``select`` then receives it as the
    keyword argument ``k_pool_normalized``.
    """
    out_dtype = q.dtype
    if q.dtype not in (torch.bfloat16, torch.float16):
        q, k_vis, v_vis = q.to(torch.bfloat16), k_vis.to(torch.bfloat16), v_vis.to(torch.bfloat16)
        if k_txt is not None:
            k_txt, v_txt = k_txt.to(torch.bfloat16), v_txt.to(torch.bfloat16)
    text_len = 0 if k_txt is None else k_txt.shape[2]
    g = geometry(latent_hw, tile, q.shape[2], k_vis.shape[2], text_len)
    tokens = fused and uses_fused(q, k_vis, v_vis, tile, (g.H, g.W))
    if qk_fp8 and (q.dtype != torch.bfloat16 or not fp8_supported(q.shape[3], tile)):
        raise ValueError(f"qk_fp8 is built for bfloat16, D = 128 and 128-token tiles (got {q.dtype}, D = {q.shape[3]}, "
                         f"tile {tuple(tile)})")
    # Q and O in token order wherever their rows can be read and written: the tiles of Q and the untile pass are for
    # other views and for grids past the kernel's 16-bit block numbers.
    _stage(events, "alloc_start")
    out = torch.empty_like(q)
    _stage(events, "alloc_end")
    rows = g.nq_blk < 65536 and (_token_rows(out) if qk_fp8 else _token_rows(q, out))
    path = ("fused" if tokens else "mixed" if rows else "tiled") + ("_fp8" if qk_fp8 else "")
    _call(path, q, k_txt, v_txt, k_vis, v_vis, out, g, select, text_len, events, balance, context, sorted_lists,
          normalize_k_pool)
    return out if out.dtype == out_dtype else out.to(out_dtype)


_CALL_PLANS = {}


def _call_plan(mode, dev, lq, lk, text_len, D, latent_hw, tile, p, default_ratio):
    """Arguments of ``li::sparse_call`` that depend on a call's sizes and parameters only (worked out once per
    configuration: every layer and step repeats it), or None for the calls it does not take.

    A configuration is looked up by the values that its parameters resolve to, read anew for each call: an absent key
    and an explicit None are not the same for all of them, and a parameter may be an object that changes in place.
    """
    H, W = latent_hw
    tt, th, tw = tile
    if not (H.__class__ is W.__class__ is tt.__class__ is th.__class__ is tw.__class__ is int):
        H, W, tt, th, tw = index(H), index(W), index(tt), index(th), index(tw)
    get, decode = p.get, mode == "decode"
    fp8 = bool(get("qk_fp8", False))
    if fp8 and not fp8_supported(D, (tt, th, tw)):
        return None
    rb, rb_key = get("row_budget"), None
    if rb is not None:
        rb = np.asarray(rb) if isinstance(rb, (list, tuple, np.ndarray)) else None
        if rb is None or rb.ndim != 1 or rb.dtype.kind not in "iub":
            return None
        rb_key = (rb.dtype.str, rb.tobytes())
    protect = get("recent_protect", 0) if decode else 0
    if protect.__class__ is not int and not isinstance(protect, Real):
        return None
    diag, sink = bool(get("force_diag", False)), bool(get("force_sink", False))
    ratio = float(get("topk_ratio", 1.0 if decode else default_ratio))
    sim = get("sim_metric", "cosine")
    metric, cos = _core.METRICS.get(sim, _lib.LI_METRIC_DOT), sim == "cosine"
    key = (decode, dev, lq, lk, text_len, D, H, W, tt, th, tw, ratio, metric, cos, protect, diag, sink, fp8, rb_key)
    plan = _CALL_PLANS.get(key)
    if plan is not None:
        return plan
    g = geometry((H, W), (tt, th, tw), lq, lk, text_len)
    n_recent = recent_blocks(p, g.tt, g.nh, g.nw, g.nk_blk) if decode else 0
    budget = _lib.LI_BUDGET_HISTORY if decode else _lib.LI_BUDGET_TOTAL
    kmax, rb_dev = _core._mask_plan(dev, g.nq_blk, g.nk_blk, g.nh, g.nw, g.num_txt_blk, n_recent, diag, sink, not decode,
                                    budget, ratio, 7, rb)
    mask = [metric, budget, 7, n_recent, diag, sink, not decode, kmax]
    plan = ([g.H, g.W, g.tt, g.th, g.tw], [int(x) for x in mask], ratio, rb_dev, fp8, cos, rb is not None)
    if len(_CALL_PLANS) >= 64:
        _CALL_PLANS.clear()
    _CALL_PLANS[key] = plan
    return plan


def native_call(mode, q, k_txt, v_txt, k_vis, v_vis, latent_hw, tile, p, default_ratio=None):
    """The whole call as one operator (``li::sparse_call``: the launches of ``sparse_attention``, with the host work
    between them in C++), or None for what it leaves to ``sparse_attention``: a context cache, element types and
    shapes that have to be converted or refused there, parameters that cannot be looked up."""
    if p.get("context_cache") is not None:
        return None
    dt, dev, shape = q.dtype, q.device, q.shape
    if (dt is not torch.bfloat16 and dt is not torch.float16) or dev.type != "cuda":
        return None
    if p.get("qk_fp8") and dt is not torch.bfloat16:
        return None
    text_len = 0 if k_txt is None else k_txt.shape[2]
    B, NH, lq, D = shape
    for t in (k_vis, v_vis, k_txt, v_txt) if text_len else (k_vis, v_vis):
        if t is None or t.dtype is not dt or t.device != dev:
            return None
        s = t.shape
        if len(s) != 4 or s[0] != B or s[1] != NH or s[3] != D:
            return None
    if k_vis.shape[2] != v_vis.shape[2] or (text_len and v_txt.shape[2] != text_len):
        return None
    try:
        plan = _call_plan(mode, dev, lq, k_vis.shape[2], text_len, D, latent_hw, tile, p, default_ratio)
    except TypeError:  # a parameter that the general route refuses or converts
        return None
    if plan is None:
        return None
    out = torch.empty_like(q)
    _core._run(_sparse_call, q, k_txt if text_len else None, v_txt if text_len else None, k_vis, v_vis, *plan, out)
    return out


def dense_attention(q, k_txt, v_txt, k_vis, v_vis):
    """The reference's dense fallback ``F.scaled_dot_product_attention(q, cat(k_txt, k_vis), cat(v_txt, v_vis))``
    (ar_sparse_operation.py:316-317, bi_sparse_operation_for_KV_cache.py:331-343, bi_sparse_operation.py:246-248).

    Runs the dense HIP kernel (li_attn_fwd_dense: every key, no concatenation formed) for fp16/bf16, D = 128 and
    visual lengths that are multiples of 4; other inputs take the reference's own torch call.
    """
    if k_txt is not None and k_txt.shape[2] == 0:
        k_txt = v_txt = None
    if _core.dense_supported(q, k_vis, v_vis, k_txt):
        return _core.attn_dense(q, k_vis, v_vis, k_txt, v_txt)
    if k_txt is not None:
        k_vis, v_vis = torch.cat([k_txt, k_vis], dim=2), torch.cat([v_txt, v_vis], dim=2)
    return F.scaled_dot_product_attention(q, k_vis, v_vis, dropout_p=0.0, is_causal=False)


def recent_blocks(params, tt, nh, nw, nk):
    """Trailing key blocks protected by ``recent_protect`` frames (ar_sparse_operation.py:263-266)."""
    rp = params.get("recent_protect", 0)
    if rp > 0:
        return min(((rp + tt - 1) // tt) * nh * nw, nk)
    return 0


def extras(params):
    """Forced-block and ragged-budget extensions (unset = the reference's rules)."""
    return dict(force_diag=bool(params.get("force_diag", False)), force_sink=bool(params.get("force_sink", False)),
                row_budget=params.get("row_budget"))

"""GPU: the entry points' one-operator call (li::sparse_call) against the general route, bit for bit, and the calls that
it leaves to that route."""
import numpy as np
import pytest
import torch

from li_sparse import ContextCache, _pipeline
from li_sparse.hy import bi_sparse_operation_for_KV_cache as hykv
from li_sparse.hy.ar_sparse_operation import run_sparse_attention
from li_sparse.hy.infer_state import get_infer_state
from li_sparse.mg import bi_sparse_operation as mgs

pytestmark = pytest.mark.gpu

CASES = [  # entry, B, H, D, dtype, (H, W), frames q / k, text, layout, params
    ("hy", 1, 3, 128, torch.bfloat16, (16, 28), 3, 6, 130, "blhd", dict(topk_ratio=0.3, recent_protect=3)),
    ("hy", 2, 2, 128, torch.float16, (16, 28), 2, 4, 128, "bhld", dict(topk_ratio=0.3, sim_metric="scaled_dot_product",
                                                                       tile_size=(2, 8, 8), force_sink=True)),
    ("hy", 1, 2, 128, torch.bfloat16, (9, 13), 3, 5, 40, "blhd", dict(sim_metric="dot", force_diag=True)),
    ("hy", 1, 2, 64, torch.bfloat16, (9, 13), 4, 4, 0, "bhld", dict(tile_size=(4, 4, 4), topk_ratio=0.25)),
    ("hy", 1, 2, 128, torch.bfloat16, (16, 28), 4, 8, 200, "blhd", dict(topk_ratio=0.4, qk_fp8=True)),
    ("hy", 1, 2, 128, torch.bfloat16, (9, 13), 4, 8, 1, "odd", dict(topk_ratio=0.4, qk_fp8=True)),
    ("hy", 1, 2, 128, torch.bfloat16, (16, 28), 2, 4, 33, "odd", dict(topk_ratio=0.4)),
    ("hy", 1, 2, 128, torch.bfloat16, (16, 28), 4, 8, 0, "blhd", dict(topk_ratio=0.2, row_budget=True)),
    ("prefill", 1, 3, 128, torch.bfloat16, (16, 28), 6, 6, 77, "blhd", dict(topk_ratio=0.2)),
    ("prefill", 1, 2, 128, torch.float16, (15, 27), 4, 4, 0, "bhld", dict(topk_ratio=0.5, force_diag=True)),
    ("mg", 1, 3, 128, torch.bfloat16, (22, 40), 4, 8, 90, "bhld", dict()),
    ("mg", 2, 2, 128, torch.bfloat16, (11, 18), 3, 3, 0, "blhd", dict(topk_ratio=0.5, sim_metric="scaled_dot_product")),
]


def _inputs(case, dev):
    _, B, NH, D, dtype, hw, fq, fk, text, layout, params = case
    gen = torch.Generator().manual_seed(3)

    def make(L):
        x = torch.randn(B, L, NH, D, generator=gen).to(dtype).to(dev).permute(0, 2, 1, 3)
        if layout == "odd":
            return torch.stack([x, x], -1)[..., 0]
        return x if layout == "blhd" else x.contiguous()

    tok = hw[0] * hw[1]
    return [make(n) for n in (fq * tok, text, text, fk * tok, fk * tok)], dict(params)


def _entry(case, x, params):
    q, kt, vt, k, v = x
    if case[0] == "mg":
        return mgs.run_sparse_attention(q, torch.cat([kt, k], 2), torch.cat([vt, v], 2), kt.shape[2], 0, case[5], params)
    if case[0] == "prefill":
        state = get_infer_state()
        state.current_chunk_index = 4
        try:
            return hykv.run_sparse_prefill_attention(q, kt, vt, k, v, 0, case[5], params)
        finally:
            state.current_chunk_index = 0
    return run_sparse_attention(q, kt, vt, k, v, 0, case[5], params)


@pytest.mark.parametrize("case", CASES)
def test_same_bits_as_the_general_route(dev, monkeypatch, case):
    print(f"[gpu] sparse_call {case}", flush=True)
    x, params = _inputs(case, dev)
    if params.get("row_budget"):
        nq = _pipeline.geometry(case[5], (4, 8, 4), x[0].shape[2], x[3].shape[2], 0).nq_blk
        params["row_budget"] = np.arange(nq) % 7 + 1
    real, taken = _pipeline.native_call, []
    monkeypatch.setattr(_pipeline, "native_call", lambda *a: taken.append(real(*a)) or taken[-1])
    a = [_entry(case, x, params) for _ in range(2)]
    monkeypatch.setattr(_pipeline, "native_call", lambda *a: None)
    b = _entry(case, x, params)
    torch.cuda.synchronize()
    assert all(t is not None for t in taken) and len(taken) == 2
    for o in a:
        assert o.dtype == b.dtype and o.stride() == b.stride()
        assert torch.equal(o.contiguous().view(torch.int16), b.contiguous().view(torch.int16))


def test_calls_left_to_the_general_route(dev):
    case = CASES[0]
    (q, kt, vt, k, v), params = _inputs(case, dev)
    call = lambda q=q, kt=kt, vt=vt, k=k, v=v, p=params, **kw: _pipeline.native_call(  # noqa: E731
        "decode", q, kt, vt, k, v, case[5], (4, 8, 4), dict(p, **kw))
    assert call() is not None
    assert call(context_cache=ContextCache()) is None
    assert call(q=q.float()) is None and call(k=k.half()) is None and call(vt=vt.half()) is None
    assert call(k=k.cpu()) is None and call(k=k[:, :2]) is None
    assert call(vt=vt[:, :, :5]) is None and call(v=v[:, :, :100]) is None
    assert call(q=q.half(), kt=kt.half(), vt=vt.half(), k=k.half(), v=v.half(), qk_fp8=True) is None
    assert call(row_budget=torch.ones(3)) is None and call(topk_ratio=[0.3]) is None
    # what these raise is the general route's own
    with pytest.raises(TypeError):
        run_sparse_attention(q, kt, vt, k.half(), v, 0, case[5], params)
    with pytest.raises(ValueError, match="row_budget has 3 entries"):
        run_sparse_attention(q, kt, vt, k, v, 0, case[5], dict(params, row_budget=[1, 2, 3]))
    with pytest.raises(KeyError):
        state = get_infer_state()
        state.current_chunk_index = 4
        try:
            hykv.run_sparse_prefill_attention(q, kt, vt, k, v, 0, case[5], {})
        finally:
            state.current_chunk_index = 0


def test_two_streams_and_threads(dev):
    """Each call's buffers are its own: calls in flight on two streams from two threads give the bits of one."""
    import threading

    case = CASES[0]
    x, params = _inputs(case, dev)
    ref = _entry(case, x, params)
    torch.cuda.synchronize()
    outs = {}

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            outs[i] = [_entry(case, x, params) for _ in range(20)]
        s.synchronize()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert all(torch.equal(o.view(torch.int16), ref.view(torch.int16)) for v in outs.values() for o in v)


@pytest.mark.parametrize("general", [False, True])
def test_budgets_outlive_a_dropped_plan(dev, monkeypatch, general):
    """The device copy of row budgets, made on one stream and read on another, is not handed out again while it is read."""
    print(f"[gpu] row budgets of a dropped plan, general={general}", flush=True)
    case = CASES[7]
    x, params = _inputs(case, dev)
    nq = _pipeline.geometry(case[5], (4, 8, 4), x[0].shape[2], x[3].shape[2], 0).nq_blk
    params["row_budget"] = [(3 * i) % 5 + 1 for i in range(nq)]
    if general:
        monkeypatch.setattr(_pipeline, "native_call", lambda *a: None)
    plans, masks = _pipeline._CALL_PLANS, _pipeline._core._MASK_PLANS
    plans.clear()
    masks.clear()
    ref = _entry(case, x, params)
    torch.cuda.synchronize()
    (_, budgets), = masks.values()
    at = budgets.data_ptr()
    del budgets
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(200_000_000)   # a bounded wait, so that the call below is still to run
        out = _entry(case, x, params)
    plans.clear()
    masks.clear()
    taken = [torch.full((nq,), 7, dtype=torch.int32, device=dev) for _ in range(64)]
    busy = not side.query()
    torch.cuda.synchronize()
    assert busy and all(t.data_ptr() != at for t in taken)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("case", [CASES[i] for i in (0, 3, 4, 6, 7, 8)])
def test_captured_call_replays(dev, case):
    """A call captured in a graph: every replay gives the bits of the eager call on the inputs that it finds."""
    print(f"[gpu] captured call {case}", flush=True)
    x, params = _inputs(case, dev)
    if params.get("row_budget"):
        nq = _pipeline.geometry(case[5], (4, 8, 4), x[0].shape[2], x[3].shape[2], 0).nq_blk
        params["row_budget"] = [(3 * i) % 5 + 1 for i in range(nq)]
    _entry(case, x, params)              # what is worked out once per configuration
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = _entry(case, x, params)
    first = [t.clone() for t in x]
    for i in range(4):
        for t, f in zip(x, first):
            t.copy_(f if i == 0 else f.roll(i, dims=2) * (1 - i / 8))
        ref = _entry(case, x, params)
        g.replay()
        got = out.clone()
        torch.cuda.synchronize()
        assert torch.equal(got.contiguous().view(torch.int16), ref.contiguous().view(torch.int16)), i
        torch.full((1 << 20,), float("nan"), device=dev)     # other work in the allocator's blocks between replays

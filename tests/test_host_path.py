"""The native host path of the fused steps (csrc/host.cpp).

It takes a call only when every check holds and otherwise returns None, so
what the Python code refuses stays refused and what it accepts stays accepted.
On the GPU its results are the Python path's, bit for bit.
"""
import pytest
import torch

DEV = "cuda"


class _Declines:
    """Stands in for the native module: every call goes to the Python code."""

    def speculative_step(self, *a):
        return None

    paged_step = speculative_step

    def prepared(self, i):
        return None


def _dense(dtype=torch.bfloat16, dev="cpu", hq=8, hkv=4, n=40, b=32, d=64, sp=8):
    gen = torch.Generator().manual_seed(3)
    q = torch.randn((hq, d), generator=gen).to(dtype)
    k = torch.randn((hkv, n, b, d), generator=gen).to(dtype)
    v = torch.randn((hkv, n, b, d), generator=gen).to(dtype)
    p = torch.stack([torch.randperm(n, generator=gen)[:sp] for _ in range(hq)]).to(torch.int32)
    return [x.to(dev) for x in (q, k, v, k.amin(2), k.amax(2), p)]


def test_declines_what_is_not_a_plain_gpu_call():
    from strict_topk import _lib
    host = _lib.host()
    a = _dense()
    assert host.speculative_step(*a, 8, False) is None            # CPU tensors
    assert host.speculative_step(*a, 8) is None                   # too few arguments
    assert host.speculative_step(None, *a[1:], 8, False) is None
    assert host.speculative_step(1, 2, 3, 4, 5, 6, 7, 8) is None
    assert host.paged_step(*[None] * 15) is None
    assert host.paged_step(*a) is None
    sparse = torch.eye(8).to_sparse()
    assert host.speculative_step(sparse, *a[1:], 8, False) is None
    nested = torch.nested.nested_tensor([torch.zeros(2, 3), torch.zeros(4, 3)])
    assert host.speculative_step(nested, *a[1:], 8, False) is None


@pytest.mark.parametrize("why", ["missing", "other torch"])
def test_without_the_module_the_python_code_runs(monkeypatch, why):
    """A process that cannot use the native module (none built for its Python, or
    one built for another torch) keeps the Python path, and its refusals."""
    import sys
    import types

    from strict_topk import _lib, step
    name = "strict_topk._host"
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setitem(sys.modules, name, None if why == "missing" else
                        types.SimpleNamespace(torch_version="0.0"))
    with pytest.warns(RuntimeWarning, match="host module not used"):
        host = _lib.host()
    assert host.speculative_step(*_dense(), 8, False) is None
    assert host.paged_step(*[None] * 15) is None and host.prepared(0) is None
    assert _lib.host() is host                                     # warned once
    with pytest.raises(ValueError, match="CUDA device"):
        step.speculative_step(*_dense(), 8)


@pytest.mark.gpu
def test_step_equals_the_python_path(monkeypatch):
    from strict_topk import _lib, step
    for hq, hkv, n, d, topk, dtype, fp32, uni in (
            (8, 4, 40, 64, 8, torch.float16, False, False), (32, 8, 300, 128, 33, torch.bfloat16,
             True, True), (64, 8, 257, 128, 20, torch.bfloat16, False, False)):
        q, k, v, lo, hi, p = _dense(dtype, DEV, hq, hkv, n, 32, d, 24)
        if fp32:
            lo, hi = lo.float(), hi.float()
        step.speculative_step(q, k, v, lo, hi, p, topk)           # the device's first call
        raw = _lib.host().speculative_step(q, k, v, lo, hi, p, topk, uni)
        assert isinstance(raw, tuple) and len(raw) == 5
        got = step.speculative_step(q, k, v, lo, hi, p, topk, union=uni)
        with monkeypatch.context() as m:
            m.setattr(_lib, "host", lambda: _Declines())
            want = step.speculative_step(q, k, v, lo, hi, p, topk, union=uni)
        for x, y in ((got.selected, want.selected), (got.output, want.output),
                     (got.state.m, want.state.m), (got.state.l, want.state.l),
                     (got.state.u, want.state.u)):
            assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)


@pytest.mark.gpu
def test_step_refuses_and_accepts_as_before():
    from torch.overrides import TorchFunctionMode

    from strict_topk import _lib, step
    q, k, v, lo, hi, p = _dense(torch.bfloat16, DEV)
    want = step.speculative_step(q, k, v, lo, hi, p, 8)
    host = _lib.host()
    for bad, msg in (
            ((q[:, :32], k, v, lo, hi, p, 8), "matching head dimensions"),
            ((q, k, v.float(), lo, hi, p, 8), "share one element dtype"),
            ((q, k.transpose(2, 3).contiguous().transpose(2, 3), v, lo, hi, p, 8), "contiguous"),
            ((q, k, v, lo[:, :-1], hi[:, :-1], p, 8), "LO/HI"),
            ((q, k, v, lo, hi.float(), p, 8), "FP32 or the element type"),
            ((q, k, v, lo, hi, p.float(), 8), "int32/int64"),
            ((q, k, v, lo, hi, p.cpu(), 8), "CUDA device")):
        assert host.speculative_step(*bad, False) is None
        with pytest.raises(ValueError, match=msg):
            step.speculative_step(*bad)
    for topk in (0, 41):
        with pytest.raises(RuntimeError, match="out of range"):
            step.speculative_step(q, k, v, lo, hi, p, topk)
    # taken by the Python code: int64 predictions, a subclass, an active mode, misalignment
    class Sub(torch.Tensor):
        pass

    shift = torch.empty(q.numel() + 1, dtype=q.dtype, device=DEV)[1:].view_as(q).copy_(q)
    for args in ((q, k, v, lo, hi, p.long(), 8), (q.as_subclass(Sub), k, v, lo, hi, p, 8),
                 (shift, k, v, lo, hi, p, 8), (q, k, v, lo, hi, p, 8.0)):
        assert host.speculative_step(*args, False) is None
        got = step.speculative_step(*args)
        assert torch.equal(torch.as_tensor(got.selected), want.selected)
        torch.testing.assert_close(got.output, want.output, rtol=3e-4, atol=3e-4)

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert host.speculative_step(q, k, v, lo, hi, p, 8, False) is None
    # another stream: ordered after its own work
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = step.speculative_step(q, k, v, lo, hi, p, 8)
    s.synchronize()
    assert torch.equal(got.output, want.output)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [True, False])
def test_paged_equals_the_python_path(monkeypatch, tokens):
    from strict_topk import _lib, paged
    gen = torch.Generator().manual_seed(5)
    caches = [tuple(torch.randn((2, n, 16, 64), generator=gen).to(torch.float16).to(DEV)
                    for _ in "kv") for n in (5, 33, 12)]
    kv = paged.pack(caches, bounds_dtype=torch.float16)
    if not tokens:
        kv.ntokens = None
    q = torch.randn((3, 4, 64), generator=gen).to(torch.float16).to(DEV)
    p = torch.randint(0, 12, (3, 4, 6), generator=gen).to(torch.int32).to(DEV)

    def calls():
        yield paged.speculative_step(q, kv, p, 7)
        yield paged.speculative_step(q, kv, p, 7, union=True)
        yield paged.exact(q, kv, 7)
        for mode, eps in (("hybrid", 0.01), ("saved", 0.0)):
            yield paged.speculative_signed_step(q, kv, p, 7, mode, 0.2, max_extra_mass=eps)

    def flat(x):
        if isinstance(x, torch.Tensor):
            return [x]
        if x is None:
            return []
        items = x if isinstance(x, tuple) else vars(x).values()
        return [t for y in items for t in flat(y)]

    got = [flat(r) for r in calls()]
    assert _lib.host().paged_step(q, kv.k_pages, kv.v_pages, kv.lo_pages, kv.hi_pages,
                                  kv.block_table, kv.nblocks, kv.ntokens, p, 7, 0, 0.0, 0.0, 0.0,
                                  0.0) is not None
    with monkeypatch.context() as m:
        m.setattr(_lib, "host", lambda: _Declines())
        want = [flat(r) for r in calls()]
    for x, y in zip(got, want):
        assert len(x) == len(y) and len(x) >= 2
        for a, b in zip(x, y):
            assert a.dtype == b.dtype and torch.equal(a, b)
    with pytest.raises(ValueError, match="topk"):
        paged.speculative_step(q, kv, p, 257)
    with pytest.raises(ValueError, match="int32"):
        paged.speculative_step(q, kv, p.long(), 7)

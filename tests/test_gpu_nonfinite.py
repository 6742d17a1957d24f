"""A predicted block that is not selected may hold anything: NaN and infinities
among its values reach neither the output of the fused steps nor that of the
repairs over saved states (zero times either would be NaN)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF, HF = torch.bfloat16, torch.float16


def _inputs(hq, hkv, n, b, d, sp, topk, dtype):
    """Inputs, the selection and predictions two thirds right, with every wrong
    block that no head of its KV head selects poisoned."""
    from strict_topk import gqa
    gen = torch.Generator(device=DEV).manual_seed(n + sp)
    q = torch.randn((hq, d), generator=gen, device=DEV, dtype=dtype)
    k = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=dtype)
    v = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=dtype)
    lo, hi = k.amin(2), k.amax(2)
    ids = gqa.select_blocks(q, lo.float(), hi.float(), topk)
    noise = torch.rand((hq, n), generator=gen, device=DEV)
    noise.scatter_(1, ids[:, : topk * 2 // 3].long(), 2.0)
    p = noise.topk(sp, dim=1).indices
    p = p.gather(1, torch.rand(p.shape, generator=gen, device=DEV).argsort(1)).to(torch.int32)
    g, bad = hq // hkv, 0
    for kv in range(hkv):
        chosen = set(ids[kv * g:(kv + 1) * g].flatten().tolist())
        wrong = [x for x in p[kv * g:(kv + 1) * g].flatten().tolist() if x not in chosen]
        for i, x in enumerate(wrong):
            v[kv, x, i % b, i % d] = (float("nan"), float("inf"), float("-inf"))[i % 3]
        bad += len(wrong)
    assert bad >= hq
    return q, k, v, lo, hi, p.contiguous(), ids, gqa.exact(q, k, v, ids)


def _same(out, want):
    assert torch.isfinite(want).all()
    torch.testing.assert_close(out, want, rtol=3e-4, atol=3e-4)


@pytest.mark.parametrize("hq,hkv,n,b,d,sp,topk,dtype", [
    (8, 8, 100, 32, 128, 12, 12, HF),      # one workgroup per head
    (32, 8, 600, 32, 128, 61, 48, BF),     # one launch, rows past SP
    (16, 8, 300, 32, 64, 64, 40, BF),
    (10, 2, 400, 16, 256, 40, 37, BF),     # two launches
    (10, 2, 400, 32, 128, 130, 37, HF),
    (10, 2, 5000, 32, 128, 50, 64, BF),    # 1024-thread tail
])
def test_steps_and_repairs_skip_unselected_blocks(hq, hkv, n, b, d, sp, topk, dtype):
    from strict_topk import gqa, gqa_light, paged, step
    q, k, v, lo, hi, p, ids, want = _inputs(hq, hkv, n, b, d, sp, topk, dtype)
    got = step.speculative_step(q, k, v, lo, hi, p, topk)
    assert torch.equal(got.selected, ids)
    _same(got.output, want)
    st = gqa.partials(q, k, v, p)
    assert not torch.isfinite(st.u).all()
    for fn in (gqa.repair_saved, gqa_light.repair_saved_light):
        _same(fn(q, k, v, ids, p, st), want)
    kv = paged.pack([(k, v)], bounds_dtype=dtype)
    _same(paged.speculative_step(q[None], kv, p[None], topk).output[0], want)


@pytest.mark.parametrize("hq,hkv,n,b,d,sp,topk,dtype", [
    (32, 8, 600, 32, 128, 61, 48, BF),
    (10, 2, 400, 16, 256, 40, 37, BF),
    (10, 2, 400, 32, 128, 130, 37, HF),
    (4, 4, 300, 32, 64, 30, 24, BF),
])
@pytest.mark.parametrize("mode,tau", [("saved", 0.0), ("hybrid", 0.0), ("hybrid", 0.03)])
def test_signed_steps_skip_unselected_blocks(hq, hkv, n, b, d, sp, topk, dtype, mode, tau):
    """With nothing low (tau = 0) no head is flagged; with poisoned low blocks the
    flagged heads' strict output is that of the selected blocks."""
    from strict_topk import paged, step
    q, k, v, lo, hi, p, ids, want = _inputs(hq, hkv, n, b, d, sp, topk, dtype)
    kv = paged.pack([(k, v)], bounds_dtype=dtype)
    one = step.speculative_signed_step(q, k, v, lo, hi, p, topk, mode, tau)
    many = paged.speculative_signed_step(q[None], kv, p[None], topk, mode, tau)
    for sel, out, bad in ((one.selected, one.result.output, one.result.fallback),
                          (many.selected[0], many.result.output[0], many.result.fallback[0])):
        assert torch.equal(sel, ids)
        _same(out, want)
        if tau == 0.0:
            assert not bad.any()

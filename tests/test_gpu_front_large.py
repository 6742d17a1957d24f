"""The fused steps' front at grid sizes past its single-item form: roles laid out
per KV row, several chunks per scoring workgroup, two slots per states wave.

A batch whose grid is large must give, request by request, the bits that the
request gives alone (a small grid): IDs, states and outputs.  The shapes sit
at the edges: rows dealt over the XCDs and not, an odd number of slots, five
query heads per KV head, one and two bounds rows per lane and pass, two and
four chunks per workgroup, requests far shorter than the table, a last block
partly filled, invalid predicted IDs and invalid pages.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF, HF = torch.bfloat16, torch.float16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from strict_topk import _lib
    _lib.lib()


def _pool(requests, hq, hkv, b, d, counts, sp, dtype, bounds, seed):
    from strict_topk.paged import PagedKV
    gen = torch.Generator(device=DEV).manual_seed(seed)
    total = hkv * sum(counts)
    kp = torch.randn((total, b, d), generator=gen, device=DEV, dtype=dtype)
    vp = torch.randn((total, b, d), generator=gen, device=DEV, dtype=dtype)
    q = torch.randn((requests, hq, d), generator=gen, device=DEV, dtype=dtype)
    order = torch.randperm(total, generator=gen, device=DEV).to(torch.int32)
    width = max(counts) + 3
    table = torch.full((requests, hkv, width), -1, dtype=torch.int32, device=DEV)
    p = torch.empty((requests, hq, sp), dtype=torch.int32, device=DEV)
    base = 0
    for r, n in enumerate(counts):
        table[r, :, :n] = order[base:base + hkv * n].view(hkv, n)
        base += hkv * n
        pick = torch.rand((hq, max(n, sp)), generator=gen, device=DEV).argsort(1)[:, :sp]
        p[r] = pick.to(torch.int32)              # past the row's end where n < sp
    p[0, :, 0] = -1
    table[requests - 1, 0, 1] = total + 7        # an invalid page
    lo, hi = kp.amin(1), kp.amax(1)
    if bounds == "fp32":
        lo, hi = lo.float(), hi.float()
    nb = torch.tensor(counts, dtype=torch.int32, device=DEV)
    part = torch.randint(1, b + 1, (requests,), generator=gen, device=DEV, dtype=torch.int32)
    return q, PagedKV(kp, vp, lo, hi, table, nb, (nb - 1) * b + part), p


def _alone(kv, r):
    from strict_topk.paged import PagedKV
    return PagedKV(kv.k_pages, kv.v_pages, kv.lo_pages, kv.hi_pages,
                   kv.block_table[r:r + 1].contiguous(), kv.nblocks[r:r + 1].contiguous(),
                   kv.ntokens[r:r + 1].contiguous())


@pytest.mark.parametrize("requests,hq,hkv,b,d,longest,sp,topk,dtype,bounds", [
    (9, 16, 2, 32, 64, 300, 121, 24, BF, "keys"),     # 18 rows, not dealt; odd slots
    (16, 40, 8, 32, 128, 200, 27, 16, HF, "fp32"),    # five heads per KV head, dealt
    (5, 8, 8, 32, 128, 2200, 4, 64, BF, "keys"),      # many chunks, two per workgroup
    (33, 8, 8, 16, 256, 500, 2, 8, BF, "fp32"),       # four chunks per workgroup, D = 256
    (9, 64, 8, 16, 128, 90, 31, 20, BF, "keys"),      # eight heads per KV head
    (3, 2, 1, 16, 64, 4500, 40, 50, BF, "keys"),      # rows of more than 4096 keys
])
def test_batch_equals_single_requests(requests, hq, hkv, b, d, longest, sp, topk, dtype, bounds):
    from strict_topk import paged
    counts = [max(1, longest * (i + 1) // requests - i % 3) for i in range(requests)]
    counts[1] = 1
    q, kv, p = _pool(requests, hq, hkv, b, d, counts, sp, dtype, bounds, 7)
    got = paged.speculative_step(q, kv, p, topk)
    sel, out = paged.exact(q, kv, topk)
    assert torch.equal(sel, got.selected)
    for r in range(requests):
        one = _alone(kv, r)
        want = paged.speculative_step(q[r:r + 1], one, p[r:r + 1].contiguous(), topk)
        for name, x, y in (("ids", got.selected, want.selected), ("m", got.state.m, want.state.m),
                           ("l", got.state.l, want.state.l), ("u", got.state.u, want.state.u),
                           ("out", got.output, want.output)):
            assert torch.equal(x[r], y[0]), (name, r, counts[r])
        torch.testing.assert_close(out[r], got.output[r], rtol=3e-4, atol=3e-4)


@pytest.mark.parametrize("hq,hkv,n,b,d,sp,topk,dtype", [
    (64, 8, 131, 32, 128, 65, 40, BF),     # eight heads per KV head, odd slots
    (40, 8, 700, 16, 256, 64, 33, HF),     # D = 256, five heads per KV head
    (24, 3, 2049, 32, 128, 100, 64, BF),   # three KV heads: rows not dealt
    (9, 1, 8000, 32, 64, 256, 200, HF),    # nine heads per KV head: the single form
])
def test_dense_front_equals_the_separate_calls(hq, hkv, n, b, d, sp, topk, dtype):
    from strict_topk import gqa, step
    gen = torch.Generator(device=DEV).manual_seed(n)
    q = torch.randn((hq, d), generator=gen, device=DEV, dtype=dtype)
    k = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=dtype)
    v = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=dtype)
    lo, hi = k.amin(2), k.amax(2)
    p = torch.rand((hq, n), generator=gen, device=DEV).argsort(1)[:, :sp].to(torch.int32)
    p = p.contiguous()
    if sp <= n:
        p[0, 0] = n + 1                      # an invalid ID
    got = step.speculative_step(q, k, v, lo, hi, p, topk)
    ids = gqa.select_blocks(q, lo.float(), hi.float(), topk)
    st = gqa.partials(q, k, v, p)
    assert torch.equal(got.selected, ids)
    for x, y in ((got.state.m, st.m), (got.state.l, st.l), (got.state.u, st.u),
                 (got.output, gqa.exact(q, k, v, ids))):
        torch.testing.assert_close(x, y, rtol=3e-4, atol=3e-4)


@pytest.mark.parametrize("d,sp,n", [
    (128, 64, 300), (128, 65, 300), (128, 128, 300), (128, 129, 300),   # 4, 8, 8, 16 row passes
    (256, 33, 200), (256, 64, 200), (256, 65, 200), (64, 129, 400), (64, 256, 400),
    (128, 40, 4096), (128, 40, 4097), (128, 129, 4097), (64, 200, 8192),  # 512 / 1024 threads
])
def test_tails_at_row_and_key_edges(d, sp, n):
    """The two-launch tails at the edges of their predicted-row passes and of
    their thread counts, against the separate calls (five query heads per KV
    head, so the one-launch step does not take the shape)."""
    from strict_topk import gqa, gqa_light, kernels, signed_fused, step
    hq, hkv, b, topk = 10, 2, 16, 37
    gen = torch.Generator(device=DEV).manual_seed(d + sp + n)
    q = torch.randn((hq, d), generator=gen, device=DEV, dtype=BF)
    k = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=BF)
    v = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=BF)
    lo, hi = k.amin(2), k.amax(2)
    ids = gqa.select_blocks(q, lo.float(), hi.float(), topk)
    noise = torch.rand((hq, n), generator=gen, device=DEV)
    noise.scatter_(1, ids[:, : topk * 2 // 3].long(), 2.0)      # two thirds predicted
    p = noise.topk(sp, dim=1).indices.to(torch.int32).contiguous()
    got = step.speculative_step(q, k, v, lo, hi, p, topk)
    st = gqa.partials(q, k, v, p)
    assert torch.equal(got.selected, ids)
    for x, y in ((got.state.u, st.u),
                 (got.output, gqa_light.repair_saved_light(q, k, v, ids, p, st)),
                 (got.output, gqa.exact(q, k, v, ids))):
        torch.testing.assert_close(x, y, rtol=3e-4, atol=3e-4)
    sg = step.speculative_signed_step(q, k, v, lo, hi, p, topk, "hybrid", 0.02)
    pred = kernels.speculate(q, k, v, p, "hybrid", 0.02, keep_mass=True)
    want = signed_fused.repair_signed_fused(q, k, v, ids, p, pred)
    assert torch.equal(sg.selected, ids)
    assert torch.equal(sg.result.positive_jobs, want.positive_jobs)
    assert torch.equal(sg.result.total_jobs, want.total_jobs)
    for x, y in ((sg.result.output, want.output), (sg.result.output, gqa.exact(q, k, v, ids)),
                 (sg.result.remaining, want.remaining)):
        torch.testing.assert_close(x, y, rtol=3e-4, atol=3e-4)


@pytest.mark.parametrize("dtype", [BF, HF])
@pytest.mark.parametrize("d,sp,n", [
    (128, 128, 300), (128, 129, 300), (128, 256, 300), (128, 200, 3000), (128, 256, 5000),
    (256, 32, 200), (256, 33, 200), (256, 64, 200), (256, 65, 200), (256, 100, 200),
    (256, 128, 200), (256, 65, 3000), (256, 33, 5000), (256, 127, 5000),
])
def test_tails_of_32_token_blocks_at_row_edges(d, sp, n, dtype):
    """The tails whose tile is 32 tokens, dense and paged, at the edges of their
    predicted-row passes and key counts, SP short of a whole pass among them:
    outputs are those of the separate calls."""
    from strict_topk import gqa, kernels, paged, signed_fused, step
    hq, hkv, b, topk = 10, 2, 32, 37
    gen = torch.Generator(device=DEV).manual_seed(d + sp + n)
    q = torch.randn((hq, d), generator=gen, device=DEV, dtype=dtype)
    k = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=dtype)
    v = torch.randn((hkv, n, b, d), generator=gen, device=DEV, dtype=dtype)
    lo, hi = k.amin(2), k.amax(2)
    ids = gqa.select_blocks(q, lo.float(), hi.float(), topk)
    noise = torch.rand((hq, n), generator=gen, device=DEV)
    noise.scatter_(1, ids[:, : topk * 2 // 3].long(), 2.0)      # two thirds predicted
    p = noise.topk(sp, dim=1).indices.to(torch.int32).contiguous()
    want = gqa.exact(q, k, v, ids)
    kv = paged.pack([(k, v)], bounds_dtype=dtype)
    one = step.speculative_step(q, k, v, lo, hi, p, topk)
    many = paged.speculative_step(q[None], kv, p[None], topk)
    for sel, out in ((one.selected, one.output), (many.selected[0], many.output[0])):
        assert torch.equal(sel, ids)
        torch.testing.assert_close(out, want, rtol=3e-4, atol=3e-4)
    for mode in ("saved", "hybrid"):
        pred = kernels.speculate(q, k, v, p, mode, 0.02, keep_mass=True)
        ref = signed_fused.repair_signed_fused(q, k, v, ids, p, pred)
        sg = step.speculative_signed_step(q, k, v, lo, hi, p, topk, mode, 0.02)
        pg = paged.speculative_signed_step(q[None], kv, p[None], topk, mode, 0.02)
        for sel, res, at in ((sg.selected, sg.result, slice(None)), (pg.selected[0], pg.result, 0)):
            assert torch.equal(sel, ids)
            for x, y in ((res.output[at], want), (res.remaining[at], ref.remaining)):
                torch.testing.assert_close(x, y, rtol=3e-4, atol=3e-4)
            for x, y in ((res.total_jobs[at], ref.total_jobs),
                         (res.positive_jobs[at], ref.positive_jobs),
                         (res.fallback[at], ref.fallback)):
                assert torch.equal(x, y)

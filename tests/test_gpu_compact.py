"""The two-launch compact speculation against the oracle: groups, capacity,
retained IDs and overflow exact, states and the low group within the
reference's tolerance (tests/check_correctness.py:22), at one slot, a full
wave of slots and one more, the widest row and one past it, capacities above
and below the high blocks, and blocks of several token chunks.
"""
import numpy as np
import pytest
import torch

from oracle import stk_oracle as O
from tests import cases as C
from tests.test_gpu_signed import _gpu, _ids  # noqa: F401

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF, HF = torch.bfloat16, torch.float16


def _inputs(hq, hkv, n, b, d, sa, sp, overlap, dtype, idtype):
    gen = torch.Generator().manual_seed(hq * 1000 + n + sp)
    q = torch.randn((hq, d), generator=gen).to(dtype)
    k = (torch.randn((hkv, n, b, d), generator=gen) * 1.2).to(dtype)
    v = torch.randn((hkv, n, b, d), generator=gen).to(dtype)
    a, p = _ids(hq, n, sa, sp, overlap, idtype, gen)
    return q, k, v, a, p


@pytest.mark.parametrize("hq,hkv,n,b,d,sp,tau,dtype,idtype", [
    (8, 8, 300, 32, 128, 64, 0.03, HF, torch.int64),
    (8, 2, 300, 32, 128, 65, 0.5, BF, torch.int32),       # capacity 3, 65 slots
    (4, 4, 400, 16, 64, 256, 0.004, BF, torch.int32),     # widest row, capacity 251
    (4, 2, 120, 48, 256, 7, 0.1, HF, torch.int32),        # three chunks per block
    (4, 4, 60, 64, 64, 1, 1.0, BF, torch.int64),          # one block, all of the mass
    (4, 4, 300, 32, 128, 257, 0.02, BF, torch.int32),     # past the two-launch form
])
def test_compact_speculation_matches_oracle(hq, hkv, n, b, d, sp, tau, dtype, idtype):
    from strict_topk.kernels import speculate
    q, k, v, _, p = _inputs(hq, hkv, n, b, d, 1, sp, 0.0, dtype, idtype)
    ref = O.speculate(C.f64(q), C.f64(k), C.f64(v), p.numpy(), "compact", tau, keep_mass=True)
    got = speculate(q.to(DEV), k.to(DEV), v.to(DEV), p.to(DEV), "compact", tau, keep_mass=True)
    assert np.array_equal(got.high.cpu().numpy(), ref.high)
    assert np.array_equal(got.overflow.cpu().numpy(), ref.overflow)
    assert np.array_equal(got.retained_ids.cpu().numpy(), ref.retained_ids)
    for name, x, y in (("m", got.state.m, ref.state.m), ("l", got.state.l, ref.state.l),
                       ("u", got.state.u, ref.state.u), ("lm", got.low.m, ref.low.m),
                       ("ll", got.low.l, ref.low.l), ("lu", got.low.u, ref.low.u),
                       ("labs", got.low_abs, ref.low_abs), ("pm", got.mass_m, ref.mass_m),
                       ("pl", got.mass_l, ref.mass_l)):
        np.testing.assert_allclose(x.cpu().double().numpy(), y, rtol=3e-4, atol=3e-4,
                                   err_msg=name)


def test_compact_speculation_ignores_an_invalid_id():
    """A predicted ID outside [0, N) has no mass: the prediction is that of the
    row without it."""
    from strict_topk.kernels import speculate
    q, k, v, _, p = _inputs(4, 2, 120, 32, 128, 1, 33, 0.0, BF, torch.int32)
    qd, kd, vd = (t.to(DEV) for t in (q, k, v))
    want = speculate(qd, kd, vd, p[:, :32].contiguous().to(DEV), "compact", 0.04)
    for bad in (-1, 120, 1 << 20):
        p[:, -1] = bad
        got = speculate(qd, kd, vd, p.to(DEV), "compact", 0.04, keep_mass=True)
        assert torch.equal(got.high[:, :32], want.high) and not got.high[:, 32].any()
        assert (got.mass_m[:, 32] == float("-inf")).all() and (got.mass_l[:, 32] == 0).all()
        assert torch.equal(got.retained_ids, want.retained_ids)
        for x, y in ((got.low.l, want.low.l), (got.low.u, want.low.u),
                     (got.low_abs, want.low_abs), (got.state.u, want.state.u)):
            torch.testing.assert_close(x, y, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("d,b", [(64, 32), (128, 32), (256, 16), (256, 64)])
def test_compact_states_are_closer_to_64_bits_than_the_saved_ones(d, b):
    """The compact states sum in short chains, as they did before they came from
    the saved states' tile: their error against the oracle is below that tile's
    on the same blocks (0.85, 0.86 and 0.70 of it at D = 64, 128 and 256)."""
    from strict_topk.kernels import speculate
    q, k, v, _, p = _inputs(8, 8, 300, b, d, 1, 64, 0.0, HF, torch.int32)
    ins = tuple(t.to(DEV) for t in (q, k, v, p))
    ref = O.block_states(C.f64(q), C.f64(k), C.f64(v), p.numpy())
    err = {}
    for mode in ("saved", "compact"):
        u = speculate(*ins, mode, 0.0).state.u.cpu().double().numpy()
        err[mode] = np.linalg.norm(u - ref.u) / np.linalg.norm(ref.u)
    assert err["compact"] < 0.95 * err["saved"], err

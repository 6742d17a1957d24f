"""The one-launch repair over every prediction mode, against the oracle.

kernels.repair, fused.repair_fused, signed_repair.repair_signed and
signed_fused.repair_signed_fused share one kernel where it covers the shape
(bf16 / fp16, D in {64, 128, 256}, B a multiple of 16, at most 256 rows).  The
oracle repairs the same prediction (as FP64), so sets, guards and budget are
exact and outputs within |err| <= 3e-4 + 3e-4 |ref| (tests/check_correctness.py:22).
The shapes are the kernel's edges: one row, a full wave of slots and one more,
256 rows, several token chunks per block, IDs past the LDS maps, retained rows
fewer and more than one pass holds, guards that flag every head.
"""
import numpy as np
import pytest
import torch

from oracle import stk_oracle as O
from tests import cases as C
from tests.test_gpu_compact import _inputs
from tests.test_gpu_signed import _gpu, _oracle_pred  # noqa: F401

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF, HF = torch.bfloat16, torch.float16

# hq, hkv, n, b, d, sa, sp, overlap, dtype, tau, eps, min_rem, tol, idtype
SHAPES = [
    (8, 8, 300, 32, 128, 64, 64, 0.8, HF, 0.03, 0.0, 1e-3, 1e-5, torch.int64),
    (8, 4, 300, 32, 128, 64, 65, 0.7, BF, 0.02, 0.05, 1e-3, 1e-5, torch.int32),   # 65 slots
    (4, 4, 200, 16, 64, 24, 100, 0.6, HF, 0.02, 0.0, 1e-3, 1e-5, torch.int64),    # SP > 64
    (8, 4, 300, 64, 128, 32, 32, 0.5, BF, 0.05, 0.01, 1e-3, 2.0, torch.int32),    # all cancel
    (8, 4, 300, 32, 128, 64, 64, 0.5, BF, 0.05, 0.0, 1.0, 1e-5, torch.int32),     # all fall back
    (4, 2, 120, 48, 256, 40, 40, 0.5, HF, 0.0, 0.0, 1e-3, 1e-5, torch.int32),     # nothing low
    (4, 1, 9000, 16, 64, 48, 48, 0.5, BF, 1.0, 0.0, 1e-3, 1e-5, torch.int64),     # past the maps
    (4, 4, 400, 32, 128, 256, 256, 0.9, BF, 0.008, 0.0, 1e-3, 1e-5, torch.int32), # widest rows
    (4, 4, 40, 32, 64, 1, 1, 0.0, BF, 0.1, 0.0, 1e-3, 1e-5, torch.int32),         # one row, missed
    # D = 256 with low hits and wrong low blocks, whole-block tiles of 16 and 32
    # tokens: compact rows of 26, 51 and 112 (four, eight and sixteen row passes)
    (4, 2, 200, 32, 256, 40, 40, 0.6, BF, 0.04, 0.0, 1e-3, 1e-5, torch.int32),
    (4, 2, 200, 32, 256, 60, 60, 0.5, HF, 0.02, 0.02, 1e-3, 1e-5, torch.int64),
    (4, 2, 300, 32, 256, 70, 128, 0.6, BF, 0.009, 0.0, 1e-3, 1e-5, torch.int32),
    (4, 2, 300, 32, 256, 70, 128, 0.6, HF, 0.009, 0.0, 1.0, 1e-5, torch.int32),   # all fall back
    (4, 2, 200, 16, 256, 40, 40, 0.6, HF, 0.04, 0.0, 1e-3, 1e-5, torch.int32),
    (4, 2, 200, 16, 256, 60, 60, 0.5, BF, 0.02, 0.0, 1.0, 1e-5, torch.int32),     # all fall back
    (4, 2, 300, 16, 256, 70, 128, 0.6, BF, 0.009, 0.01, 1e-3, 1e-5, torch.int64),
    (4, 4, 300, 32, 128, 64, 200, 0.6, BF, 0.006, 0.0, 1e-3, 1e-5, torch.int32),  # 167 rows
]


@pytest.mark.parametrize("mode", ["saved", "hybrid", "compact"])
@pytest.mark.parametrize("shape", SHAPES)
def test_repairs_match_oracle(shape, mode):
    from strict_topk import fused, kernels, signed_fused, signed_repair
    hq, hkv, n, b, d, sa, sp, overlap, dtype, tau, eps, min_rem, tol, idtype = shape
    q, k, v, a, p = _inputs(hq, hkv, n, b, d, sa, sp, overlap, dtype, idtype)
    qd, kd, vd, ad, pd = (t.to(DEV) for t in (q, k, v, a, p))
    pred = kernels.speculate(qd, kd, vd, pd, mode=mode, mass_threshold=tau, keep_mass=True)
    opred = _oracle_pred(pred)
    if mode == "compact":
        opred.retained_ids = pred.retained_ids.cpu().numpy()
    qn, kn, vn = (C.f64(t) for t in (q, k, v))
    an, pn = a.numpy(), p.numpy()
    flagged = False
    for name, gpu, ref in (
            ("split", kernels.repair, O.repair), ("fused", fused.repair_fused, O.repair_fused),
            ("signed", signed_repair.repair_signed, O.repair_signed),
            ("signed_fused", signed_fused.repair_signed_fused, O.repair_signed_fused)):
        more = () if name == "split" else (eps,)
        want = ref(qn, kn, vn, an, pn, opred, min_rem, tol, *more)
        got = gpu(qd, kd, vd, ad, pd, pred, min_rem, tol, *more)
        what = (name, mode, shape)
        assert got.fallback.cpu().numpy().tolist() == want.fallback.tolist(), what
        np.testing.assert_allclose(got.remaining.cpu().double().numpy(), want.remaining,
                                   rtol=1e-4, atol=1e-6, err_msg=str(what))
        if more and eps > 0:
            assert got.approximate_heads.cpu().numpy().tolist() == want.approximate_heads.tolist()
            np.testing.assert_allclose(got.extra_mass_bound.cpu().double().numpy(),
                                       want.extra_mass_bound, rtol=1e-4, atol=1e-7)
        if name.startswith("signed"):
            assert got.positive_jobs.cpu().numpy().tolist() == want.positive_jobs.tolist(), what
            assert got.total_jobs.cpu().numpy().tolist() == want.total_jobs.tolist(), what
        m = C.error_metrics(C.f64(got.output), want.output)
        assert m["passed"], (what, m)
        flagged = flagged or bool(got.fallback.any())
    if min_rem == 1.0 and mode != "saved":
        assert flagged


def test_fallback_streams_tiles_when_a_state_is_not_finite():
    """A kept prediction row that is not finite flags its head, whose output is
    then recomputed from the selected blocks' tiles."""
    from strict_topk import fused, kernels
    q, k, v, a, p = _inputs(4, 4, 100, 32, 128, 24, 24, 0.8, BF, torch.int32)
    qd, kd, vd, ad, pd = (t.to(DEV) for t in (q, k, v, a, p))
    want = O.exact_attention(C.f64(q), C.f64(k), C.f64(v), a.numpy())
    for mode in ("hybrid", "compact"):
        pred = kernels.speculate(qd, kd, vd, pd, mode=mode, mass_threshold=0.0)
        pred.state.u[:, :, 5] = float("nan")
        for fn in (kernels.repair, fused.repair_fused):
            got = fn(qd, kd, vd, ad, pd, pred)
            assert got.fallback.all()
            m = C.error_metrics(C.f64(got.output), want)
            assert m["passed"], (mode, fn.__name__, m)


REPAIRS = ("split", "fused", "signed", "signed_fused")


def _repair(name):
    from strict_topk import fused, kernels, signed_fused, signed_repair
    return {"split": (kernels.repair, O.repair), "fused": (fused.repair_fused, O.repair_fused),
            "signed": (signed_repair.repair_signed, O.repair_signed),
            "signed_fused": (signed_fused.repair_signed_fused, O.repair_signed_fused)}[name]


def _check(name, ins, pred, opred, min_rem, tol, eps):
    """One repair against the oracle's on the same prediction."""
    q, k, v, a, p = ins
    gpu, ref = _repair(name)
    more = () if name == "split" else (eps,)
    want = ref(C.f64(q), C.f64(k), C.f64(v), a.numpy(), p.numpy(), opred, min_rem, tol, *more)
    got = gpu(*(t.to(DEV) for t in ins), pred, min_rem, tol, *more)
    what = (name, pred.mode, eps)
    assert got.fallback.cpu().numpy().tolist() == want.fallback.tolist(), what
    np.testing.assert_allclose(got.remaining.cpu().double().numpy(), want.remaining, rtol=1e-4,
                               atol=1e-6, err_msg=str(what))
    if more and eps > 0:
        assert got.approximate_heads.cpu().numpy().tolist() == want.approximate_heads.tolist()
        np.testing.assert_allclose(got.extra_mass_bound.cpu().double().numpy(),
                                   want.extra_mass_bound, rtol=1e-4, atol=1e-7)
    m = C.error_metrics(C.f64(got.output), want.output)
    assert m["passed"], (what, m)
    return want


@pytest.mark.parametrize("mode", ["saved", "hybrid", "compact"])
@pytest.mark.parametrize("d,b,sp,slot", [
    (128, 32, 24, 0),      # row 0, which rows past SP repeat
    (128, 32, 24, 17),
    (64, 16, 200, 130),    # sixteen row passes
    (256, 32, 40, 0),
])
def test_rows_that_are_not_kept_add_nothing(d, b, sp, slot, mode):
    """A predicted block that is not selected may hold anything: with NaN and an
    infinity among its values the repairs give what the oracle gives, with the
    oracle's flags."""
    from strict_topk.kernels import speculate
    h = 4
    q, k, v, a, p = _inputs(h, h, 260, b, d, 24, sp, 0.7, BF, torch.int32)
    for i in range(h):
        chosen = set(a[i].tolist())
        wrong = [j for j in range(sp) if int(p[i, j]) not in chosen]
        j = wrong[0] if slot == 0 else min(wrong, key=lambda x: abs(x - slot))
        if slot == 0:
            p[i, [0, j]] = p[i, [j, 0]]
            j = 0
        v[i, int(p[i, j]), 3, 7] = float("inf") if i % 2 else float("nan")
        v[i, int(p[i, j]), 1, 9] = float("-inf")
    ins = (q, k, v, a, p)
    for tau in (0.0, 0.05):
        pred = speculate(*(t.to(DEV) for t in (q, k, v, p)), mode=mode, mass_threshold=tau,
                         keep_mass=True)
        opred = _oracle_pred(pred)
        if mode == "compact":
            opred.retained_ids = pred.retained_ids.cpu().numpy()
        for name in REPAIRS:
            with np.errstate(invalid="ignore"):
                want = _check(name, ins, pred, opred, 1e-3, 1e-5, 0.01 if mode != "saved" else 0.0)
            assert np.isfinite(want.output).all()
            if tau == 0.0:
                assert not want.fallback.any()


@pytest.mark.parametrize("mode", ["hybrid", "compact"])
@pytest.mark.parametrize("d,b,idtype", [(128, 32, torch.int32), (64, 64, torch.int64),
                                        (256, 16, torch.int32)])
def test_fallback_is_the_selected_blocks_alone(d, b, idtype, mode):
    """A flagged head's output comes from the selected blocks, each slot once:
    neither a block predicted twice nor a prediction whose kept states are no
    longer those of the query changes it."""
    from strict_topk.kernels import speculate
    h, n, sa, sp = 4, 9000 if d == 64 else 120, 40, 40
    q, k, v, a, p = _inputs(h, h, n, b, d, sa, sp, 0.7, BF, idtype)
    for i in range(h):
        # a selected block predicted twice (and an invalid selected ID below)
        hits = [j for j in range(sp) if (a[i] == p[i, j]).any()]
        p[i, hits[1]] = p[i, hits[0]]
    a[:, -1] = -1
    ins = (q, k, v, a, p)
    exact = O.attention(C.f64(q), C.f64(k), C.f64(v), a[:, :-1].numpy())
    for stale in (False, True):
        pred = speculate(*(t.to(DEV) for t in (q, k, v, p)), mode=mode, mass_threshold=0.02,
                         keep_mass=True)
        if stale:
            pred.state.u.mul_(-1.5)
            pred.state.m.add_(0.25)
        for name in REPAIRS:
            # every fraction is below it
            got = _repair(name)[0](*(t.to(DEV) for t in ins), pred, 2.0, 1e-5)
            assert got.fallback.any()
            flagged = got.fallback.cpu().numpy()
            m = C.error_metrics(C.f64(got.output)[flagged], exact[flagged])
            assert m["passed"], (name, mode, stale, m)

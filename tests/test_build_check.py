"""The build's check of the generated code (build_lib.misplaced_copies): register
copies ahead of a join's exec restore are found, and the forms in which a copy
belongs under the branch's mask are not."""
import importlib.util
from pathlib import Path

import pytest


def _check(body):
    path = Path(__file__).resolve().parents[1] / "strict-topk-overlap_amd" / "build_lib.py"
    spec = importlib.util.spec_from_file_location("build_lib", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module.misplaced_copies(["_Z1kv:", *body.strip("\n").split("\n")])


BRANCH = """
\ts_and_saveexec_b64 s[2:3], s[38:39]
\ts_cbranch_execz .LBB0_2
; %bb.1:
\tv_mov_b32_e32 v47, v1
"""


@pytest.mark.parametrize("copy", [
    "v_mov_b32_e32 v167, v189", "v_mov_b64_e32 v[2:3], v[4:5]", "v_accvgpr_write_b32 a0, v1",
    "scratch_store_dword off, v162, off offset:4", "scratch_load_dword v34, off, off offset:4"])
def test_a_copy_ahead_of_the_restore_is_found(copy):
    bad = _check(BRANCH + f".LBB0_2:\n\t{copy}\n\ts_mov_b64 s[56:57], s[18:19]\n"
                 "\ts_or_b64 exec, exec, s[2:3]\n")
    assert len(bad) == 1 and copy in bad[0] and "_Z1kv" in bad[0]


def test_a_join_without_a_label_is_checked():
    bad = _check("\ts_and_saveexec_b64 s[2:3], vcc\n; %bb.1:\n\tv_mov_b32_e32 v1, v9\n"
                 "; %bb.2:\n\tv_mov_b32_e32 v4, v5\n\ts_or_b64 exec, exec, s[2:3]\n")
    assert len(bad) == 1 and "v4, v5" in bad[0]


@pytest.mark.parametrize("body", [
    # after the restore
    BRANCH + ".LBB0_2:\n\ts_or_b64 exec, exec, s[2:3]\n\tv_mov_b32_e32 v167, v189\n",
    # a body that was moved away and is entered under its mask
    ".LBB0_7:\n\tv_mov_b32_e32 v98, v101\n\ts_or_b64 exec, exec, s[2:3]\n"
    "\ts_cbranch_execnz .LBB0_7\n",
    # a body that ends with its own restore
    "\ts_and_saveexec_b64 s[4:5], vcc\n\ts_cbranch_execz .LBB0_9\n; %bb.3:\n"
    "\tv_mov_b32_e32 v5, v6\n\ts_or_b64 exec, exec, s[4:5]\n",
    # lanes of a register that exec does not mask, and constants
    BRANCH + ".LBB0_2:\n\tv_writelane_b32 v255, s88, 29\n\tv_mov_b32_e32 v3, 0\n"
    "\ts_or_b64 exec, exec, s[2:3]\n"])
def test_copies_under_their_own_mask_pass(body):
    assert _check(body) == []

"""Waits that count loads hold in the compiler's assembly of this source (llmp_amd/csrc/check_counted_waits.py, also a step
of the build), and the check sees a wait that is one short. Needs hipcc, no GPU; fails, not skips, where hipcc is missing."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def module():
    spec = importlib.util.spec_from_file_location(
        "check_counted_waits", os.path.join(ROOT, "llmp_amd", "csrc", "check_counted_waits.py"))
    loaded = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(loaded)
    assert os.path.exists(loaded.HIPCC), "hipcc is missing: the waits cannot be checked"
    return loaded


def test_counted_waits_hold_on_every_path(module):
    assert module.check() >= 5


@pytest.mark.parametrize("left,weights,holds", [(9, 4, True), (9, 3, False), (1, 0, True)])
def test_a_wait_that_counts_loads_that_are_not_there_is_found(module, left, weights, holds):
    """A loop of one input and `weights` other loads a chunk: an input is needed at the second barrier after it."""
    body = "\n".join(
        ["\ts_waitcnt vmcnt(0)", "\ts_barrier", ".LBB0_1:", f"\ts_waitcnt vmcnt({left})", "\ts_barrier", "\t;;#ASMSTART",
         "\tglobal_load_lds_dwordx4 v1, s[0:1]", "\t;;#ASMEND"] + ["\tglobal_load_dword v2, v3, off"] * weights +
        ["\ts_cbranch_scc1 .LBB0_1", "\ts_waitcnt vmcnt(0)", "\ts_endpgm"])
    if holds:
        module.check_panel("kernel", body)
    else:
        with pytest.raises(AssertionError, match="loads to LDS may still"):
            module.check_panel("kernel", body)

"""Waits that count loads hold in the compiler's assembly of this source (llmp_amd/csrc/check_counted_waits.py, also a step
of the build), and the check sees a wait that is one short. Needs hipcc, no GPU; fails, not skips, where hipcc is missing."""
import importlib.util
import os
import re

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
    assert module.check() >= 53


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


def test_the_reconstructions_words_are_where_they_are_read(module):
    """Up to five bits a value a lane's states lie in the two words that it holds, always in the same order: nothing is
    chosen at run time. Chosen by branches, a pair for each of sixteen tiles (which the compiler made of a third register),
    they cost the unfused reconstruction 2 to 3 us of 40; by selects 0.5."""
    kernels = list(module.kernels_of(module.assembly_of("exl3.hip"), r"Reconstruct\w*KernelILi[012]ELi[12345]E"))
    assert len(kernels) >= 45  # three codebooks by five rates: transposed, and the weights themselves both ways
    for name, body in kernels:
        decode = body[body.find("ds_write"):body.rfind("ds_write")]
        assert "s_cbranch_execz" not in decode and decode.count("v_cndmask") < 32, name  # (the signs of H take some)


def test_only_the_wide_products_transform_asks_for_the_grid(module):
    """The transform that lays its result out for the product of many rows needs the grid's size, which comes with 256 bytes
    of arguments; the others take their own, fewer than 128 bytes, and no more."""
    described = module.assembly_of("exl3.hip").split("amdhsa.kernels:")[1].split("- .agpr_count:")[1:]
    sizes = [int(re.search(r"\.kernarg_segment_size: (\d+)", d).group(1)) for d in described
             if re.search(r"\.name: +\S*HadamardKernelILi[01]ELi[01]ELb0E", d)]
    assert len(sizes) >= 3 and max(sizes) < 128, sizes


@pytest.mark.parametrize("between,holds", [("v_add_f32_e32 v5, v1, v2", True), ("v_mov_b32_e32 v8, v1", False),
                                           ("v_mov_b32_e32 v1, v7", False), ("ds_read_b32 v7, v2", False)])
def test_a_register_named_while_a_load_to_it_is_on_its_way_is_found(module, between, holds):
    """Past the loop, two loads whose results nothing reads any more, before the waits that close it."""
    body = "\n".join(
        [".LBB0_1:", "\ts_waitcnt vmcnt(0) lgkmcnt(0)", "\t;;#ASMSTART", "\tglobal_load_dwordx2 v[7:8], v[2:3], off",
         "\t;;#ASMEND", "\ts_cbranch_scc1 .LBB0_1", "\t" + between, "\ts_waitcnt vmcnt(0)", "\ts_endpgm"])
    if holds:
        module.check_registers("kernel", body)
    else:
        with pytest.raises(AssertionError, match="on its way"):
            module.check_registers("kernel", body)


@pytest.mark.parametrize("ahead,loop,holds", [
    (3, "load vm2 lgkm ask", True),
    (3, "load vm3 lgkm ask", False),  # a wait one short
    (3, "vm2 lgkm ask load", False),  # the next stage asked for behind the words: the wait counts a load that is not there
    (4, "load vm3 lgkm ask", False),  # a stage filled while it is read
])
def test_a_stage_asked_for_before_it_landed_is_found(module, ahead, loop, holds):
    """A ring of one load a stage whose words are asked for a step ahead of their use, in the loop's order and in others."""
    ask = "\n".join(["\t;;#ASMSTART\n\tds_read_b32 v1, v2\n\t;;#ASMEND"] * module.ASK_LEAST)
    text = {"load": "\tglobal_load_lds_dwordx4 v[2:3], off", "vm2": "\ts_waitcnt vmcnt(2)", "vm3": "\ts_waitcnt vmcnt(3)",
            "lgkm": "\ts_waitcnt lgkmcnt(0)", "ask": ask}
    body = "\n".join([text["load"]] * ahead + [f"\ts_waitcnt vmcnt({ahead - 1})", ask, ".LBB0_1:"] + [text[w] for w in loop.split()] +
                     ["\ts_cbranch_scc1 .LBB0_1", "\ts_waitcnt vmcnt(0) lgkmcnt(0)", "\ts_endpgm"])
    if holds:
        module.check_ring("kernel", body, 1)
    else:
        with pytest.raises(AssertionError, match="words"):
            module.check_ring("kernel", body, 1)


def test_the_packed_products_loads_keep_their_places_among_the_compilers():
    """Their waits count the ring's loads, which the compiler may move, with those written as instructions: each of these, and
    the wait for LDS, says that it touches memory, so that nothing moves across it."""
    with open(os.path.join(ROOT, "llmp_amd", "csrc", "exl3.hip")) as f:
        written = re.findall(r'asm volatile\("(?:global_load|s_waitcnt)[^;]*;', f.read())
    assert len(written) >= 3 and all('"memory"' in w for w in written), written

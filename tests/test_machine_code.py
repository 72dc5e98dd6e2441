"""What inline assembly leaves to the kernels' author, checked on the built library's machine code (see isa.py)."""
import os
import re

import pytest

import isa

needs_objdump = pytest.mark.skipif(not os.path.exists(isa.OBJDUMP), reason="no llvm-objdump")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    from lv_xattn import _lib
    _lib.load()
    return isa.functions(_lib.LIB_PATH, str(tmp_path_factory.mktemp("code")))


@needs_objdump
def test_mfma_results_have_their_wait_states(kernels):
    assert sum(any(i.op.startswith("v_mfma") for i in body) for body in kernels.values()) > 50
    early = {name: found for name, found in ((n, isa.mfma_results_touched_early(b)) for n, b in kernels.items()) if found}
    assert not early, {name: found[:2] for name, found in early.items()}


@needs_objdump
def test_loads_to_lds_wait_for_m0(kernels):
    assert sum(any(isa.to_lds(i) for i in body) for body in kernels.values()) > 50
    early = {name: found for name, found in ((n, isa.m0_used_early(b)) for n, b in kernels.items()) if found}
    assert not early, (len(early), {name: found[:2] for name, found in list(early.items())[:4]})


@needs_objdump
def test_addresses_that_come_out_of_lanes_have_their_wait_states(kernels):
    early = {name: found for name, found in ((n, isa.scalars_used_early(b)) for n, b in kernels.items()) if found}
    assert not early, {name: found[:2] for name, found in early.items()}


@needs_objdump
def test_registers_that_assembly_loads_are_left_alone_until_the_wait(kernels):
    """fwd_few_kernel requests Q by inline assembly long before it waits for it: no path of the built code may copy,
    spill or use those registers in between.  Its wait is one statement: everything, or, in waves that have requested two
    pieces of K and V behind Q, all but those.  Which waves these are cannot be seen in the code's paths; that the number
    is that of the two requests can."""
    few = {n: b for n, b in kernels.items() if "fwd_few_kernel" in n}
    assert len(few) == 16
    for name, body in few.items():
        request = next(i for i, ins in enumerate(body) if ins.op == "global_load_dwordx4")
        jump = next(i for i, ins in enumerate(body) if ins.target and "LVX_FEW_TWO" in ins.args[0])
        all_of_it, but_two_pieces = body[jump + 1:jump + 3]
        assert all_of_it.op == but_two_pieces.op == "s_waitcnt" and body[jump].target == but_two_pieces.addr, name
        assert isa.waits_for(all_of_it) == 0, name
        assert isa.waits_for(but_two_pieces) == sum(isa.to_lds(i) for i in body[request:jump]), name
        assert not isa.loads_touched_early(body, stated=[but_two_pieces]), name


@needs_objdump
def test_a_bias_on_its_way_is_left_alone_until_the_wait(kernels):
    """The forward with a dense bias requests it by inline assembly a tile ahead: the same."""
    biased = {n: b for n, b in kernels.items() if re.search(r"fwd_kernelILi\d+ELb[01]ELb1E", n)}
    assert len(biased) == 16
    for name, body in biased.items():
        assert not isa.loads_touched_early(body), name


PLANTED = """
0000000000001000 <kernel>:
\tv_mfma_f32_32x32x16_bf16 v[4:19], v[20:23], v[82:85], 0    // 000000001000: D3B58004 02
\ts_cbranch_vccnz 2                                         // 000000001008: BF870002 <kernel+0x14>
\ts_nop 11                                                  // 00000000100C: BF80000B
\tv_mov_b32_e32 v4, 0                                       // 000000001010: 7E080280
\tv_max3_f32 v2, v30, v5, v6                                // 000000001014: D1D30002
\ts_endpgm                                                  // 00000000101C: BF810000
"""


def test_the_check_takes_every_path():
    (body,) = isa.parse(PLANTED).values()
    (found,) = isa.mfma_results_touched_early(body)
    assert found[1].op == "v_max3_f32" and found[2] == 1
    (body,) = isa.parse(PLANTED.replace("BF870002", "BF87FFFD")).values()      # the branch goes back instead
    assert [x[1].op for x in isa.mfma_results_touched_early(body)] == []


def test_a_copy_of_a_register_in_flight_is_found():
    text = PLANTED.replace("v_mfma_f32_32x32x16_bf16 v[4:19], v[20:23], v[82:85], 0    ", "global_load_dwordx4 v[4:7], v[20:21], off    ")
    (body,) = isa.parse(text).values()
    assert sorted(x[1].op for x in isa.loads_touched_early(body)) == ["v_max3_f32", "v_mov_b32"]
    (body,) = isa.parse(text.replace("s_nop 11 ", "s_waitcnt vmcnt(0) ").replace("v5, v6", "v8, v9")).values()
    assert not isa.loads_touched_early(body)


IN_FLIGHT = """
0000000000001000 <kernel>:
\tglobal_load_dwordx4 v[4:7], v[20:21], off                  // 000000001000: DD5C8000 02
\ts_cbranch_vccnz 3                                         // 000000001008: BF870003 <kernel+0x18>
\tglobal_load_lds_dwordx4 v8, s[4:5]                        // 00000000100C: DDF48000 02
\ts_nop 0                                                   // 000000001014: BF800000
\tglobal_load_lds_dwordx4 v8, s[4:5] offset:1024            // 000000001018: DDF48400 02
\ts_waitcnt vmcnt(1)                                        // 000000001020: BF8C0F71
\tv_mov_b32_e32 v9, v5                                      // 000000001024: 7E120305
\ts_endpgm                                                  // 000000001028: BF810000
"""


def test_a_wait_that_leaves_the_load_in_flight_is_none():
    def early(text):
        (body,) = isa.parse(text).values()
        return [x[1].op for x in isa.loads_touched_early(body)], body
    assert early(IN_FLIGHT)[0] == []                        # one load at least stands behind it
    assert early(IN_FLIGHT.replace("vmcnt(1)", "vmcnt(2)"))[0] == ["v_mov_b32"]       # one path has one only
    assert early(IN_FLIGHT.replace("BF870003", "BF870005"))[0] == ["v_mov_b32"]       # none
    (body,) = isa.parse(IN_FLIGHT.replace("vmcnt(1)", "vmcnt(2)")).values()
    assert not isa.loads_touched_early(body, stated=[body[5]])


def test_a_load_to_lds_right_behind_m0_is_found():
    text = PLANTED.replace("v_mov_b32_e32 v4, 0  ", "s_add_i32 m0, s50, 0x400  ")
    for load in ("global_load_lds_dwordx4 v8, s[4:5] offset:16  ", "buffer_load_dwordx4 v8, s[4:7], s9 offen lds  "):
        (body,) = isa.parse(text.replace("v_max3_f32 v2, v30, v5, v6  ", load)).values()
        assert [x[1].addr for x in isa.m0_used_early(body)] == [0x1014]
        (body,) = isa.parse(text.replace("s_nop 11  ", load)).values()       # before the write, a branch over it
        assert not isa.m0_used_early(body)


def test_an_address_right_out_of_a_lane_is_found():
    text = PLANTED.replace("v_mfma_f32_32x32x16_bf16 v[4:19], v[20:23], v[82:85], 0  ", "v_readlane_b32 s5, v30, 7  ")
    text = text.replace("v_max3_f32 v2, v30, v5, v6  ", "global_load_lds_dwordx4 v8, s[4:5]  ")
    (body,) = isa.parse(text).values()
    (found,) = isa.scalars_used_early(body)
    assert found[1].addr == 0x1014 and found[2] == 1
    (body,) = isa.parse(text.replace("s_cbranch_vccnz 2  ", "s_nop 4  ")).values()
    assert not isa.scalars_used_early(body)

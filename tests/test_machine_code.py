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
def test_the_form_that_folds_its_own_parts_leaves_them_alone_too(kernels):
    """fwd_fewest_kernel: the same, its count requested in front of Q, and the parts that are read back."""
    fewest = {n: b for n, b in kernels.items() if "fwd_fewest_kernel" in n}
    assert len(fewest) == 16
    for name, body in fewest.items():
        jump = next(i for i, ins in enumerate(body) if ins.target and "LVX_FEW_TWO" in ins.args[0])
        assert next(i for i, ins in enumerate(body) if ins.op == "global_load_dwordx2") < \
            next(i for i, ins in enumerate(body) if ins.op == "global_load_dwordx4"), name
        assert isa.waits_for(body[jump + 1]) == 0 and not isa.loads_touched_early(body, stated=[body[jump + 2]]), name


@needs_objdump
def test_a_bias_on_its_way_is_left_alone_until_the_wait(kernels):
    """The forward with a dense bias requests it by inline assembly a tile ahead: the same."""
    biased = {n: b for n, b in kernels.items() if re.search(r"fwd_kernelILi\d+ELb[01]ELb1E", n)}
    assert len(biased) == 16
    for name, body in biased.items():
        assert not isa.loads_touched_early(body), name


RING = "LVX_DQ_MORE"       # the wait of dq_kernel and dq_few_kernel


@needs_objdump
def test_stages_of_dS_on_their_way_are_left_alone_until_the_wait(kernels):
    """dq_kernel and dq_few_kernel request dS^T by inline assembly into 64 to 96 registers, stages ahead of their use.  A
    stage is four loads of dS^T and, by 4 KB of a work-group or 1 KB of a wave, those of 32 rows of K."""
    checked = 0
    for name, body in kernels.items():
        m = re.search(r"dq_(few_)?kernelILi(\d+)E", name)
        if not m:
            continue
        found, stages, left = isa.ring_loads_touched_early(body, RING)
        row_bytes = 2 * max(64, int(m.group(2)))
        loads = 4 + 32 * row_bytes // (1024 if m.group(1) else 4096)
        assert stages == (4 if m.group(1) else 5 if row_bytes == 256 else 6) and left == (stages - 2) * loads, name
        assert not found, (name, found[:2])
        checked += 1
    assert checked == 64


@needs_objdump
@pytest.mark.parametrize("form", ["dq_kernelILi128E", "dq_few_kernelILi64E"])
def test_what_would_touch_a_stage_on_its_way_is_found(kernels, form):
    name = next(n for n in kernels if form in n)
    body = kernels[name]
    waits = [i for i, ins in enumerate(body) if ins.target is not None and RING in ins.args[0]]

    def found(changed):
        return isa.ring_loads_touched_early([changed.get(i, ins) for i, ins in enumerate(body)], RING)[0]
    left = isa.waits_for(body[waits[0] + 2])
    of_k = left // (len(waits) - 2) - 4                         # requested behind a stage's dS^T
    late = lambda n: {w + 2: isa.Ins(body[w + 2].addr, "s_waitcnt", [f"vmcnt({left + n})"]) for w in waits}
    assert not found(late(of_k)) and found(late(of_k + 1))      # one load too few is waited for
    load = next(ins for i, ins in enumerate(body) if i > waits[0] and ins.op == "buffer_load_dwordx4")     # of step 0, for step R - 1
    register = "v" + re.match(r"v\[(\d+):", load.args[0]).group(1)
    for w, early in ((waits[1], True), (waits[-1], False)):     # a copy behind a wait for an earlier stage, and behind its own
        at = next(i for i in range(w + 3, w + 60) if body[i].op.startswith("v_") and body[i].target is None)
        copy = found({at: isa.Ins(body[at].addr, "v_mov_b32", ["v0", register])})
        assert any(x[1].op == "v_mov_b32" for x in copy) == early, (at, copy[:2])


@needs_objdump
def test_only_a_forward_that_folds_takes_the_arguments_of_the_fold(tmp_path):
    """What every launch copies and fetches: a decoded token's two launches are as long as the host takes to queue them."""
    from lv_xattn import _lib
    _lib.load()
    size = {n: b for n, b in isa.argument_bytes(_lib.LIB_PATH, str(tmp_path)).items() if re.search("fwd_(few_|wide_)?kernel", n)}
    folding = {n for n in size if re.search(r"fwd_wide_kernelILi\d+ELb[01]ELb[01]ELb1E", n)}
    assert len(folding) == 8 and len(size) > 40
    assert len({size[n] for n in folding}) == len({size[n] for n in size.keys() - folding}) == 1
    assert min(size[n] for n in folding) > max(size[n] for n in size.keys() - folding)


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

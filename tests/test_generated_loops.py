"""The hand-scheduled loops under csrc/ are generated text that is committed: every .inc file must be
what its generator writes today (the generators also lint their own output for the instruction
hazards the assembler does not resolve, and refuse to write a stream that has one)."""
import importlib.util
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "lv-xattn_amd", "csrc")


def _generated():
    spec = importlib.util.spec_from_file_location("lvx_build", os.path.join(ROOT, "lv-xattn_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod.GENERATED


@pytest.mark.parametrize("script,args,out", _generated(), ids=[g[2] for g in _generated()])
def test_committed_loop_is_what_its_generator_writes(script, args, out):
    env = {k: v for k, v in os.environ.items() if not k.startswith("LVX_")}      # no experiment switches
    r = subprocess.run([sys.executable, os.path.join(CSRC, script), *args], capture_output=True, text=True, env=env)
    assert r.returncode == 0, r.stderr
    assert r.stdout == open(os.path.join(CSRC, out)).read(), f"{out} is stale: run lv-xattn_amd/build.py"
    body = r.stdout.splitlines()
    assert body[0].startswith("// generated by") and all(l.startswith('"') and l.endswith('\\n"') for l in body[1:])


def test_every_included_loop_has_a_generator():
    listed = {g[2] for g in _generated()}
    on_disk = {f for f in os.listdir(CSRC) if f.endswith(".inc")}
    assert on_disk == listed
    for f in os.listdir(CSRC):
        if f.endswith(".hip"):
            text = open(os.path.join(CSRC, f)).read()
            for inc in listed:
                if inc.split("_loop")[0] in f.replace(".hip", "") and f'#include "{inc}"' not in text:
                    pytest.fail(f"{inc} is generated but {f} does not include it")


@pytest.mark.parametrize("out", [g[2] for g in _generated() if g[0] == "gen_bwd_loop.py" and g[1][0] == "p"])
def test_backward_loop_reads_a_ring_behind_the_wait_of_its_loads(out):
    """P-waves: what an LDS read takes out of the Q and dO rings was requested before a count of loads in flight that
    covers it, with a barrier behind that count (vector-memory operations complete in issue order).  Of a wave that requests
    no metadata, the one with the fewest operations behind a load, over the prologue and three trips."""
    text = [l[1:-3] for l in open(os.path.join(CSRC, out)).read().splitlines()[1:]]
    top, end = text.index("LVX_BWD_LOOP_%=:"), next(i for i, l in enumerate(text) if l.startswith("s_sub_i32 s64"))
    issued, m0, load_of, waited, safe, checked = 0, 0, {}, 0, 0, 0
    skip = None
    for line in text[:top] + 3 * text[top + 1:end]:
        if skip:
            skip = None if line == skip else skip
            continue
        op, _, rest = line.partition(" ")
        if op == "s_cbranch_scc1" and "NOMETA" in rest:
            skip = rest + ":"
        elif op == "s_add_i32" and rest.startswith("m0, s62"):
            m0 = int(rest.split(",")[2])
        elif rest.startswith("m0,"):
            m0 = None                       # of the metadata, or of the bias (below)
        elif op.startswith("global_load_lds_dwordx4") or op.startswith("global_store"):
            issued += 1
            if "lds" in op and m0 is not None:
                load_of.setdefault(m0 // 8192, []).append(issued)
        elif op == "s_waitcnt" and "vmcnt" in rest:
            waited = max(waited, issued - int(re.search(r"vmcnt\((\d+)\)", rest).group(1)))
        elif op == "s_barrier":
            safe = waited
        elif op.startswith("ds_read"):
            addr = re.search(r", v(\d+)", rest)
            at = int(addr.group(1))
            if 200 <= at <= 215:            # row reads from the Q ring, transposing reads from the dO ring
                off = re.search(r"offset:(\d+)", rest)
                ring = (int(off.group(1)) if off else 0) // 8192 + (6 if at >= 208 else 0)
                assert all(n <= safe for n in load_of.get(ring, [])), (line, ring, load_of[ring], safe)
                checked += ring in load_of
    assert checked > 50


@pytest.mark.parametrize("out", [g[2] for g in _generated() if g[0] == "gen_bwd_loop.py" and "bias" in g[1]])
def test_backward_loop_with_a_bias_reads_it_behind_the_wait_of_its_loads(out):
    """The one LDS tile of a wave's bias: what is read of it was requested in the step before and waited for by a count of loads
    in flight, and a step's request follows a wait for the last read of the tile it replaces (LDS operations
    complete in order, as vector-memory operations do; no other wave touches the tile)."""
    text = [l[1:-3] for l in open(os.path.join(CSRC, out)).read().splitlines()[1:]]
    top, end = text.index("LVX_BWD_LOOP_%=:"), next(i for i, l in enumerate(text) if l.startswith("s_sub_i32 s64"))
    assert "s_waitcnt vmcnt(0)" in text[:top]           # what was requested in front of the loop: the first tile of the bias among it
    lines = text[:top] + 3 * text[top + 1:end]

    def walk(lines):
        issued = lds = waited = read_until = last_read = 0
        bias, seen, reads, skip, tile = [], [], 0, None, False
        for line in lines:
            if skip:
                skip = None if line == skip else skip
                continue
            op, _, rest = line.partition(" ")
            if op == "s_cbranch_scc1" and "NOMETA" in rest:
                skip = rest + ":"
            elif rest.startswith("m0,"):
                tile = "s39" in rest
            elif op.startswith("global_"):
                issued += 1
                if tile and "lds" in op:
                    assert last_read <= read_until, (line, last_read, read_until)
                    bias.append(issued)
                    tile = False
            elif op == "s_waitcnt" and "vmcnt" in rest:
                waited = max(waited, issued - int(re.search(r"vmcnt\((\d+)\)", rest).group(1)))
            elif op == "s_waitcnt":
                read_until = max(read_until, lds - int(re.search(r"lgkmcnt\((\d+)\)", rest).group(1)))
            elif op.startswith("ds_"):
                lds += 1
                if re.search(r", v233\b", rest):
                    assert all(n <= waited for n in bias), (line, bias[-4:], waited)
                    seen.append(len(bias))
                    last_read, reads = lds, reads + 1
        return seen, reads
    seen, reads = walk(lines)
    assert reads == 3 * 6 * 8 and seen == [4 * (k // 8) for k in range(reads)]      # 8 reads a step, of the 4 loads before
    # a count one too high, a request in front of the wait for the reads: found
    for old, new in (("s_waitcnt vmcnt(6)", "s_waitcnt vmcnt(7)"), ("s_waitcnt lgkmcnt(4)", "s_waitcnt lgkmcnt(5)")):
        assert old in lines
        with pytest.raises(AssertionError):
            walk([new if l == old else l for l in lines])


@pytest.mark.parametrize("out", [g[2] for g in _generated() if g[0] == "gen_fwd_loop_wide.py" and "bias" in g[1]])
def test_forward_loop_with_a_bias_reads_it_behind_the_wait_of_its_loads(out):
    """As above: all 16 loads of a tile are waited for by count before the first read of it, a refill follows a wait for the last read,
    and in front of a tile's barrier the count covers every load of K and V."""
    text = [l[1:-3] for l in open(os.path.join(CSRC, out)).read().splitlines()[1:]]
    top, end = text.index("LVX_FWDW_LOOP_%=:"), text.index("s_branch LVX_FWDW_LOOP_%=")
    lines = text[:top] + 3 * text[top + 1:end]

    def walk(lines):
        issued = lds = waited = read_until = last_read = 0
        bias, tiles, seen = [], [], []
        for line in lines:
            op, _, rest = line.partition(" ")
            if op.startswith("global_load") or op.startswith("buffer_load"):
                issued += 1
                if op.startswith("buffer"):
                    assert last_read <= read_until, line
                    bias.append(issued)
                elif "lds" in op:
                    tiles.append(issued)
            elif op == "s_waitcnt" and "vmcnt" in rest:
                waited = max(waited, issued - int(re.search(r"vmcnt\((\d+)\)", rest).group(1)))
            elif op == "s_waitcnt":
                read_until = max(read_until, lds - int(re.search(r"lgkmcnt\((\d+)\)", rest).group(1)))
            elif op == "s_barrier" and seen:
                assert tiles[-1] <= waited
            elif op.startswith("ds_"):
                lds += 1
                if re.search(r", v245\b", rest):
                    assert all(n <= waited for n in bias), (line, bias[-4:], waited)
                    seen.append(len(bias))
                    last_read = lds
        return seen
    seen = walk(lines)
    assert seen == [16 * (1 + k // 16) for k in range(7 * 16)]       # the prologue's tile and two a trip
    kv = 8 if "_128" in out else 4
    for old, new in ((f"s_waitcnt vmcnt({kv})", f"s_waitcnt vmcnt({kv + 1})"), ("s_waitcnt lgkmcnt(0)", "s_waitcnt lgkmcnt(1)")):
        assert old in lines
        with pytest.raises(AssertionError):
            walk([new if l == old else l for l in lines])

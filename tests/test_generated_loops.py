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

"""Writes the hand-scheduled body of the 256-row GEMM tiles (lvx_gemm.hip, gemm_tile_kernel):

    python gen_gemm_loop.py p|t p|t 256|128 256|224 > lvx_gemm_loop_<A><B>_<TN>_<TM>.inc

p: the operand is stored [row][k], read with 16-byte LDS reads; t: stored [k][row], read with transposing
LDS reads.  The tile is 256 x TN, four waves (2 x 2) of 128 x TN / 2, each with its SIMD to itself: the
accumulators (16 registers per 32 x 32) live in accumulation registers, and a wave's operands serve
twice the MFMAs per LDS byte that eight waves' would.  A tile of 224 rows x 256 has its waves side by side, 224 x 64
each (seven blocks of rows do not halve): nine operands for 14 MFMAs where the others have eight for 16.

One statement runs all stages (64 values of k each) of a tile, one or more, and leaves the C tile in LDS as
16-bit values.  A stage is 64 deep because a piece of an operand stored [row][k] is then 128 bytes of
a row, a whole cache line: with 32 the same loads touch twice the lines and a 256 x 128 tile of such operands
ran at 880 TFLOP/s where one of [k][row] operands ran at 1290.
Stage s of A is in ring slot s % 3, of B in slot s % NSB: with a 256 x 256 tile two slots for B are what
fits beside three for A (160 KiB), which is the operand that streams from HBM (the other is shared
by the tiles of an XCD and comes from its L2).  With two slots for both, 64 KiB in flight per CU, the loads
and LDS reads without any MFMA took 655 us of a product of 838; with the third, 549 of 820.
Per k-step of 16 a wave issues its MFMAs from one operand set and between them the LDS reads of the next
k-step into the other.  One barrier per stage, in front of its last k-step: by then every wave has read
all of stage s, whose slots may now be overwritten - by B of stage s + NSB in that k-step and A of stage
s + 3 in the next - and its own wait has seen its part of stage s + 1 land, which is read from there on.
Loads are buffer loads: what lies past the end of the contraction is out of the descriptor's range and
arrives as zeros.

Registers (must match the asm statement in lvx_gemm.hip):
  v[0:63] two operand sets   v[64:79] byte offsets of this wave's pieces (A, then B)   v[80:95] the same for
  the last stage   v[96:107] A read addresses, four per slot   v[108:119] the same for B
  v120 address of this lane's first piece of the C tile   v[121:136] those of its pieces
  a[16 (WM nt + mt) :] accumulators   224 rows: v[122:129] the operands that do not fit v[0:63]
  s[40:43], s[44:47] descriptors of A, B   s48, s49 bytes per stage   s50 LDS address of this wave's part of slot
  0   s51 stages left to run   s52, s60 stages of A, B to request after the next   s53, s54 offset of the next
  stage in A, B   s55, s61 stages to request before the second pair of operands (0: none)   s[56:57],
  s[58:59] its bases
The text names the MFMA and the conversion by the macros LVX_GEMM_MFMA and LVX_GEMM_CVT.
"""
import os
import sys

# experiment switches (comma separated in LVX_GEMM_OPTS); none is set in a normal build
OPTS = set(o for o in os.environ.get("LVX_GEMM_OPTS", "").split(",") if o)
AT, BT, TN, TM = sys.argv[1] == "t", sys.argv[2] == "t", int(sys.argv[3]), int(sys.argv[4])
assert TM == 256 or (TM == 224 and TN == 256 and not AT)
WM, WN = (4, TN // 64) if TM == 256 else (7, 2)
NSA, NSB = 3, 2 if TN == 256 else 3
UNROLL = 6 if NSB == 2 else 3
A_BYTES, B_BYTES = TM * 128, TN * 128
NLA, NLB = TM // 32, TN // 32              # 1 KiB pieces per wave and stage
NL = NLA + NLB
OPER, VOFF, VTAIL, RA, RB, EP, EPA = 0, 64, 80, 96, 108, 120, 121
MFMA, CVT = '" LVX_GEMM_MFMA "', '" LVX_GEMM_CVT "'


def vr(base, n):
    return f"v[{base}:{base + n - 1}]"


def ar(base, n):
    return f"a[{base}:{base + n - 1}]"


def am(s, mt):
    return OPER + 32 * s + 4 * mt


def bn(s, nt):
    if TM == 224:
        return OPER + 32 * s + 28 if nt == 0 else 122 + 4 * s
    return OPER + 32 * s + 16 + 4 * nt


def reads(u, kk, s):
    """LDS reads of k-step kk of stage u into operand set s, in the order the MFMAs want them."""
    def one(trans, r, dst, t, rows):
        if trans:       # address per 32-row tile; a k-step is 16 rows of `rows` values further down
            o = kk * 16 * rows * 2
            return [f"ds_read_b64_tr_b16 {vr(dst, 2)}, v{r + t} offset:{o}",
                    f"ds_read_b64_tr_b16 {vr(dst + 2, 2)}, v{r + t} offset:{o + 4 * rows * 2}"]
        return [f"ds_read_b128 {vr(dst, 4)}, v{r + kk} offset:{t * 4096}"]

    out = []
    for nt in range(WN):
        out += one(BT, RB + 4 * (u % NSB), bn(s, nt), nt, TN)
        if nt == 0:
            for mt in range(WM):
                out += one(AT, RA + 4 * (u % NSA), am(s, mt), mt, TM)
    return out


def request(which, u):
    """This wave's pieces of A or B of stage u, the next one to be requested: the write of M0 and the load, which
    needs a wait state behind it."""
    out = []
    for j in range(NLA if which == "a" else NLB):
        if which == "a":
            dst, v, src = (u % NSA) * A_BYTES + j * 4096, VOFF + j, "s[40:43], s53"
        else:
            dst, v, src = NSA * A_BYTES + (u % NSB) * B_BYTES + j * 4096, VOFF + NLA + j, "s[44:47], s54"
        out.append([f"s_add_i32 m0, s50, {dst}", f"buffer_load_dwordx4 v{v}, {src} offen lds"])
    return out


SLOW = []
N_LABEL = [0]


def advance(which):
    """The source of A or B moves to the next stage unless it stands at the last."""
    N_LABEL[0] += 1
    n = N_LABEL[0]
    left, off, step, seg, base, first, v0, nl = (("s52", "s53", "s48", "s55", "s[40:41]", "s[56:57]", 0, NLA) if which == "a" else
                                                 ("s60", "s54", "s49", "s61", "s[44:45]", "s[58:59]", NLA, NLB))
    SLOW.extend([f"LVX_GEMM_SEG{n}_%=:", f"s_mov_b64 {base}, {first}", f"s_mov_b32 {off}, 0",
                 f"s_branch LVX_GEMM_SAME{n}_%=", f"LVX_GEMM_LAST{n}_%=:"])
    SLOW.extend(f"v_mov_b32 v{VOFF + v0 + j}, v{VTAIL + v0 + j}" for j in range(nl))
    SLOW.append(f"s_branch LVX_GEMM_STAY{n}_%=")
    return [f"s_cmp_eq_u32 {left}, 0", f"s_cbranch_scc1 LVX_GEMM_STAY{n}_%=", f"s_sub_u32 {left}, {left}, 1",
            f"s_add_u32 {off}, {off}, {step}", f"s_sub_u32 {seg}, {seg}, 1", f"s_cmp_eq_u32 {seg}, 0",
            f"s_cbranch_scc1 LVX_GEMM_SEG{n}_%=", f"LVX_GEMM_SAME{n}_%=:", f"s_cmp_eq_u32 {left}, 0",
            f"s_cbranch_scc1 LVX_GEMM_LAST{n}_%=", f"LVX_GEMM_STAY{n}_%=:"]


def kstep(s, rd, rq, tail):
    """The MFMAs of operand set s with the reads `rd` and requests `rq` between them; M0 is written before an MFMA
    and the load follows behind it."""
    out = []
    n = WM * WN
    rd, rq = list(rd), list(rq)
    span = n - n // 4               # the reads are out by three quarters of the k-step
    nr, nq = len(rd), len(rq)
    k = 0
    for nt in range(WN):
        for mt in range(WM):
            a = 16 * (WM * nt + mt)
            loads = []
            for _ in range(nq * (k + 1) // n - nq * k // n):
                m0, load = rq.pop(0)
                loads += [load] if not loads else [m0, "s_nop 0", load]
                out += [m0] if len(loads) == 1 else []
            out.append(f"{MFMA} {ar(a, 16)}, {vr(bn(s, nt), 4)}, {vr(am(s, mt), 4)}, {ar(a, 16)}")
            for _ in range(nr * min(k + 1, span) // span - nr * min(k, span) // span):
                out.append(rd.pop(0))
            out += loads
            k += 1
    assert not rd and not rq
    return out + tail


def stage(u):
    """Stage s with s % UNROLL == u.  Its first k-step requests A of stage s + 2."""
    in_flight = NLA if NSB == 2 else NL     # what has been requested after the stage that has to be there
    out = ["s_waitcnt lgkmcnt(0)"] + kstep(0, reads(u, 1, 1), request("a", u + 2), advance("a"))
    out += ["s_waitcnt lgkmcnt(0)"] + kstep(1, reads(u, 2, 0), [], [])
    out += ["s_waitcnt lgkmcnt(0)"] + kstep(0, reads(u, 3, 1), [], [])
    out += ["s_waitcnt lgkmcnt(0)", f"s_waitcnt vmcnt({in_flight})", "s_barrier"]
    out += kstep(1, reads(u + 1, 0, 0), request("b", u + NSB), advance("b"))
    out += ["s_sub_u32 s51, s51, 1", "s_cmp_eq_u32 s51, 0", "s_cbranch_scc1 LVX_GEMM_END_%="]
    return out


def main():
    lines = []
    zero = [f"v_accvgpr_write_b32 a{r}, 0" for r in range(16 * WM * WN)]
    for u in range(NSB):            # B of stages 0 .. NSB - 1, A of stages 0 and 1
        for which in ("a", "b") if u < 2 else ("b",):
            for m0, load in request(which, u):
                lines += [m0, zero.pop(0), load]
            lines += advance(which)
    lines += zero
    lines += [f"s_waitcnt vmcnt({NL + (NLB if NSB == 3 else 0)})", "s_barrier"] + reads(0, 0, 0)
    lines += ["LVX_GEMM_LOOP_%=:"]
    for u in range(UNROLL):
        lines += stage(u)
    lines += ["s_branch LVX_GEMM_LOOP_%="] + SLOW
    # the C tile goes to LDS: piece (nt, vg) of a row is 4 columns, 8 bytes
    lines += ["LVX_GEMM_END_%=:", "s_waitcnt vmcnt(0)", "s_waitcnt lgkmcnt(0)", "s_barrier", "s_nop 15", "s_nop 3"]
    for c in range(4 * WN):
        lines.append(f"v_xor_b32 v{EPA + c}, {c * 16}, v{EP}")
    group = 0
    in_reach = 65536 // (32 * TN * 2)       # blocks of rows an instruction's offset reaches
    for m0 in range(0, WM, in_reach):
        for nt in range(WN):
            for vg in range(4):
                if m0:
                    lines.append(f"v_add_u32 v{EPA + 4 * nt + vg}, 0x10000, v{EPA + 4 * nt + vg}")
                for mt in range(m0, min(WM, m0 + in_reach)):
                    t = 4 * (group % 16)
                    group += 1
                    a = 16 * (WM * nt + mt) + 4 * vg
                    lines += [f"v_accvgpr_read_b32 v{t + i}, a{a + i}" for i in range(4)]
                    lines += [f"{CVT} v{t}, v{t}, v{t + 1}", f"{CVT} v{t + 1}, v{t + 2}, v{t + 3}",
                              f"ds_write_b64 v{EPA + 4 * nt + vg}, {vr(t, 2)} offset:{(mt - m0) * 32 * TN * 2}"]
    lines += ["s_waitcnt lgkmcnt(0)"]
    for x, y in zip(lines, lines[1:]):
        if x.startswith("s_add_i32 m0") and y.startswith("buffer_load"):
            raise SystemExit(f"hazard: {y} right behind the write of M0")
    if "nodma" in OPTS:
        lines = [l for l in lines if not l.startswith("buffer_load") and not l.startswith("s_add_i32 m0")]
    if "nolds" in OPTS:
        lines = [l for l in lines if not l.startswith("ds_read")]
    if "nobar" in OPTS:
        lines = [l for l in lines if l != "s_barrier"]
    if "nomfma" in OPTS:
        lines = [l for l in lines if not l.startswith(MFMA)]
    print("// generated by gen_gemm_loop.py - do not edit")
    for l in lines:
        print(f'"{l}\\n"')


main()

"""Writes the hand-scheduled steady-state loops of the gfx950 backward kernel (lvx_bwd.hip):

    python gen_bwd_loop.py p bf16 128 plain > lvx_bwd_loop_p_bf16_128_plain.inc   (P-waves: S, P = exp2(..), dV^T)
    python gen_bwd_loop.py d bf16 128 > lvx_bwd_loop_d_bf16_128.inc               (D-waves: dP, dS, dK^T)

for bf16 and f16, head dimensions 128 and 64, and P-waves without ("plain") and with ("masked") key
intervals per row, the latter also with a dense bias ("bias").  Each is one inline-asm statement with every register named here.  One trip does six steps (the
six tile buffers of each ring and the two-deep P / dS^T buffers then sit at immediate offsets);
the first step of a trip is a step i with i % 6 == 3.  Inside a step the 16 MFMAs of a wave (8 with heads of 64) are
spread over its other instructions (LDS operand reads eight operands ahead, the exponentials or
the dS arithmetic of an earlier tile, the global -> LDS loads and the dS^T copy-out), so that a
wave keeps the matrix pipe fed by itself.

LDS map in bytes (lvx_bwd.hip): Q ring 6 x 8192 at 0, dO ring at 49152, dS^T tiles 2 x 8192 at
98304, P hand-over 2 x 8192 at 114688; the metadata of a tile, 6 x 768 bytes, is a separate array: 256 bytes
of LSE and delta, with intervals per row 256 each of starts and ends (32 rows, twice).

The last tile of a head may have fewer than 32 rows: when the walk comes to it, the lanes' load offsets are
replaced by ones whose rows are clamped to the window's last (RAGGED, out of line), and restored with the
next head.  Masked: a step asks with one compare per lane whether any
row of the tile cuts the wave's 32 tokens and only then goes through the out-of-line block that zeroes
the hidden elements of P.

Bias: 32 rows x the wave's 32 tokens of fp32, 4 KiB in an LDS tile of its own that no other wave touches.  In the second
half of step i the bias of tile i is read from there into the registers that the bias of tile i-1 had, and
behind those reads the four loads of tile i+1's are requested, a whole step before they are waited for.  A lane's
loads would be 16 of 4 bytes per tile (two rows of 32 tokens each), four times as many as the tile's own.  An LDS row of 128
bytes is 32 tokens of row 8 n + 4 (s & 1) + (s >> 1) for slot s of the n-th load: the lane's 16 rows are 256 bytes
apart, and the two halves of a wave in different banks.

Registers, both roles: v[0:63] resident accumulators (dV^T / dK^T)   v[64:95] resident B operands
(K rows / V rows)   v[96:111], v[112:127] the two score sets (raw S / dP), swapping every step
v[128:159] eight operand slots  v[200:207] row-read addresses into "its" ring (P: Q, D: dO)
v[208:215] transposing-read addresses into the other ring.   s40 scale*log2(e) (P) / scale (D)
P-waves: v[168:175] P packed   v[176:191] LSE*log2(e) of 16 rows   v[192:199] dS^T copy-out data
  v216 P hand-over write address   v217 metadata read address   v218, v219 dS^T copy-out read addresses (transposing
  reads: four tokens of a row each)   v220 copy-out global offset   v221..v224 global offsets of the four tile loads   v225 of
  the metadata load   v226, v227 rows by which the lane's two rows of a head's last tile are past the window
  v229 scratch   masked: v228 read address of the interval of row lane % 32   v229, v230 that interval
  v231 the lane's token, out of every interval if it is past the sample   v232 bytes by which the lane's row of
  a head's last tile is past the window, in the waves that fetch intervals
  s41 / s42 bytes per Q / dO tile   s[44:45] Q, s[46:47] dO, s[48:49] metadata, s[50:51] dS^T
  workspace address of the next tile to request   s52 tiles left in its head   s53 tiles per head
  s[54:55] / s[56:57] / s[60:61] what a head change adds to the Q / dO / workspace address
  s62 LDS address of this wave's part of Q buffer 0   s63 of the metadata records   s64 trips
  s65 1 in the waves that request metadata: wave 0 LSE and delta, wave 1 interval starts, wave 2 ends
  s[66:77] workspace addresses of the tiles in flight   s[78:79], s[88:89] scratch
  s[80:81] what a head change adds to the metadata address   s82 1 if the last tile of a head has clamped
  rows, else -1   s83 / s84 bytes per Q / dO row   masked: s85 bytes of metadata per tile   s86 first token of the wave, s87 one
  past its last   s[90:91] all ones if not all of them exist   s92 1 if dS^T leaves as streaming stores
  bias: v[234:249] the bias of 16 rows   v233 its read address   v250 the lane's row in the first of a tile's four loads
  v251 bytes of its chunk in a row   s39 LDS address of the tile   s93 bytes per row   s94 per 32 rows   s95 log2(e)
  s[96:97] address of the next tile to request (its first row, token 0)   s98 tiles left in its head   s99 last row of a
  head's last tile   s[100:101] what a head change adds
D-waves: v[168:175] P handed over   v[176:183] dS packed   v[184:199] delta*scale of 16 rows
  v216 P hand-over read address   v217 metadata read address   v218, v223..v225 dS^T staging write addresses, one per
  group of four rows
"""
import os
import re
import sys

# experiment switches (comma separated in LVX_GEN_OPTS); none is set in a normal build
OPTS = dict((o.split("=") + ["1"])[:2] for o in os.environ.get("LVX_GEN_OPTS", "").split(",") if o)
ROLE = sys.argv[1] if len(sys.argv) > 1 else "p"
for _o in list(OPTS):      # a switch for one role only: p_novalu, d_nolds, ...
    if _o.startswith(ROLE + "_"):
        OPTS[_o[2:]] = OPTS[_o]
F16 = len(sys.argv) > 2 and sys.argv[2] == "f16"
DH = int(sys.argv[3]) if len(sys.argv) > 3 else 128
BIAS = len(sys.argv) > 4 and sys.argv[4] == "bias"
MASKED = BIAS or len(sys.argv) > 4 and sys.argv[4] == "masked"
MFMA = "v_mfma_f32_32x32x16_f16" if F16 else "v_mfma_f32_32x32x16_bf16"
CVT = "v_cvt_pk_f16_f32" if F16 else "v_cvt_pk_bf16_f32"
NKK, NDT = DH // 16, DH // 32           # k-steps of S / dP, 32-wide blocks of dV^T / dK^T
NOP = NKK + 2 * NDT                     # MFMAs of a step, one LDS operand each

ACC, BREG, SET, STG, RA, TA = 0, 64, (96, 112), 128, 200, 208
NSLOT, AHEAD = 8, 7
TILE_B, DO_RING, DST_B, DST_SZ, PB_SZ, META_SZ = 8192, 49152, 98304, 8192, 8192, 768
# P role
PU, LSE, CPD = 168, 176, 192
A_PB, A_META, A_CP, G_CP, G_DMA, G_META = 216, 217, (218, 219), 220, 221, 225
EXCESS, A_IV, IV, TOKEN = 226, 228, 229, 231
IV_EXCESS = 232
BV, A_BV, BROW, BCHUNK = 234, 233, 250, 251
# D role
DSU, DELTA, TMP, A_DS = 176, 184, 219, (218, 223, 224, 225)


def vr(base, n=1):
    return f"v{base}" if n == 1 else f"v[{base}:{base + n - 1}]"


def sr(base, n=1):
    return f"s{base}" if n == 1 else f"s[{base}:{base + n - 1}]"


class Stream:
    """Instruction list with a model of the in-order LDS queue for s_waitcnt lgkmcnt."""

    def __init__(self, seed=None):
        self.out = []
        self.n_lds = 0
        self.tag = {}
        self.done = 0           # LDS operations 1 .. done are known to have completed
        self.last_write = 0     # position of the last ds_write
        if seed is not None:    # what the step before left in flight: see carry_over()
            self.n_lds = seed["n"]
            self.tag = dict(seed["tag"])

    def emit(self, s):
        if "nodma" in OPTS and (s.startswith("global_load_lds") or s.startswith("s_add_i32 m0")):
            return
        if "nostore" in OPTS and s.startswith("global_store"):
            return
        if "novalu" in OPTS and s.startswith("v_") and not s.startswith("v_mfma"):
            return
        if "nomfma" in OPTS and s.startswith("v_mfma"):
            return
        if "nobar" in OPTS and s.startswith("s_barrier"):
            return
        self.out.append(s)

    def lds(self, text, tag=None):
        if "nolds" in OPTS and "_tr_" in text or "nolds" in OPTS and text.startswith("ds_read_b128 v[1") and int(text.split("[")[1].split(":")[0]) < 160:
            text = None
        if text is not None:
            self.out.append(text)
        self.n_lds += 1
        if tag is not None:
            self.tag[tag] = self.n_lds
        if text is not None and text.startswith("ds_write"):
            self.last_write = self.n_lds

    def wait(self, tag):
        if self.tag[tag] <= self.done:      # an earlier wait of this step covers it
            return
        n = min(self.n_lds - self.tag[tag], 15)
        self.out.append(f"s_waitcnt lgkmcnt({n})")
        self.done = self.n_lds - n

    def carry_over(self, u_next):
        """What a step leaves to the next one: the LDS operations it issued after its last write (the
        next step waits at its top until only these are in flight: LDS operations complete in order, so
        the writes other waves are about to read have then landed) and, among them, the reads of the
        first operands of the next step."""
        done = self.last_write
        if BIAS:        # more reads than can be counted, but their last ones were waited for behind the writes
            done = max(done, self.done)
        n = self.n_lds - done
        tag = {t: pos - done for t, pos in self.tag.items()     # <= 0: read before the write
               if isinstance(t, tuple) and t[0] == "op" and t[1] == u_next}
        assert len(tag) == AHEAD and n <= 15, (n, tag)
        return {"n": n, "tag": tag}

    def wait_needed(self, tag):
        return self.n_lds - self.tag[tag]


def spread(st, mfmas, side, shares):
    """Emit MFMA k (a callable writing its wait + instruction), then shares[k] entries of side."""
    pos = 0
    for k, m in enumerate(mfmas):
        m()
        take = shares[k] if k + 1 < len(mfmas) else 10 ** 6
        while take > 0 and pos < len(side):
            x = side[pos]
            pos += 1
            if isinstance(x, list):     # a branch and what it jumps over stay together
                for y in x:
                    st.emit(y)
                take -= len(x)
            else:
                x() if callable(x) else st.emit(x)
                take -= 1
    assert pos == len(side), (pos, len(side))


def p_read_op(st, u, n):
    """LDS read of operand n of P-wave step u: Q rows of tile i (k-step n), then dO^T of tile i-1."""
    sl_i, sl_p = (u + 3) % 6, (u + 2) % 6
    slot = STG + 4 * (n % NSLOT)
    if n < NKK:
        st.lds(f"ds_read_b128 {vr(slot, 4)}, v{RA + n} offset:{sl_i * TILE_B}", ("op", u, n))
    else:
        j, dt = (n - NKK) // NDT, (n - NKK) % NDT
        off = sl_p * TILE_B + j * 4096
        st.lds(f"ds_read_b64_tr_b16 {vr(slot, 2)}, v{TA + 2 * dt} offset:{off}")
        st.lds(f"ds_read_b64_tr_b16 {vr(slot + 2, 2)}, v{TA + 2 * dt + 1} offset:{off}", ("op", u, n))


def p_fetch(u, ahead):
    """Request of tile i + ahead by a P-wave in step u, and the walk to the tile after it.  A load to LDS needs a
    wait state behind the write of M0: a part of the walk, which for Q and the metadata is over by then."""
    sl_f = (u + 3 + ahead) % 6
    ws_new = 66 + 2 * sl_f
    f = [[f"s_add_i32 m0, s63, {sl_f * META_SZ}", "s_cmp_eq_u32 s65, 0", f"s_cbranch_scc1 LVX_BWD_NOMETA{u}{ahead}_%=",
          f"global_load_lds_dword v{G_META}, s[48:49]", f"LVX_BWD_NOMETA{u}{ahead}_%=:"]]
    walk = [[f"s_mov_b64 {sr(ws_new, 2)}, s[50:51]"], ["s_add_u32 s50, s50, 8192", "s_addc_u32 s51, s51, 0"],
            ["s_add_u32 s48, s48, s85", "s_addc_u32 s49, s49, 0"], ["s_add_u32 s44, s44, s41", "s_addc_u32 s45, s45, 0"]]
    for n, (base, src) in enumerate(((0, "s[44:45]"), (1024, "s[44:45]"), (DO_RING, "s[46:47]"), (DO_RING + 1024, "s[46:47]"))):
        f += [f"s_add_i32 m0, s62, {sl_f * TILE_B + base}", *walk[n], f"global_load_lds_dwordx4 v{G_DMA + n}, {src}"]
    f += ["s_add_u32 s46, s46, s42", "s_addc_u32 s47, s47, 0",
          ["s_sub_i32 s52, s52, 1", "s_cmp_lg_u32 s52, 0", f"s_cbranch_scc1 LVX_BWD_SAMEHEAD{u}{ahead}_%=",
           "s_add_u32 s44, s44, s54", "s_addc_u32 s45, s45, s55", "s_add_u32 s46, s46, s56", "s_addc_u32 s47, s47, s57",
           "s_add_u32 s48, s48, s80", "s_addc_u32 s49, s49, s81",
           "s_add_u32 s50, s50, s60", "s_addc_u32 s51, s51, s61", "s_mov_b32 s52, s53",
           "s_cmp_eq_u32 s82, 1", f"s_cbranch_scc1 LVX_BWD_WHOLE{u}{ahead}_%=", f"LVX_BWD_SAMEHEAD{u}{ahead}_%=:",
           "s_cmp_eq_u32 s52, s82", f"s_cbranch_scc1 LVX_BWD_RAGGED{u}{ahead}_%=", f"LVX_BWD_WALKED{u}{ahead}_%=:"]]
    return f


def p_ragged(u, ahead):
    """Out of line: the tile the walk has come to is a head's last and has clamped rows, so that the lanes'
    load offsets go back by the rows they are too far; or a head with such a tile begins, and they return."""
    def move(op):
        return [x for n in range(4) for x in (f"v_mul_lo_u32 v{IV}, v{EXCESS + n % 2}, s{83 + n // 2}",
                                              f"{op} v{G_DMA + n}, v{G_DMA + n}, v{IV}")] \
            + ([f"{op} v{G_META}, v{G_META}, v{IV_EXCESS}"] if MASKED else [])
    return [f"LVX_BWD_WHOLE{u}{ahead}_%=:", *move("v_add_u32"), f"s_branch LVX_BWD_SAMEHEAD{u}{ahead}_%=",
            f"LVX_BWD_RAGGED{u}{ahead}_%=:", *move("v_sub_u32"), f"s_branch LVX_BWD_WALKED{u}{ahead}_%="]


def p_store(hint):
    return [f"global_store_dwordx4 v{G_CP}, {vr(CPD, 4)}, s[78:79]{hint}", f"global_store_dwordx4 v{G_CP}, {vr(CPD + 4, 4)}, s[78:79] offset:1024{hint}"]


def p_keep(u):
    """Out of line: the launch's dS^T fits the memory-side cache and is stored without the streaming hint."""
    return [f"LVX_BWD_KEEP{u}_%=:", *p_store(""), f"s_branch LVX_BWD_STORED{u}_%="]


def p_mask(u):
    """Out of line: some row of tile i-1 cuts this wave's tokens.  P's elements outside their row's interval
    become 0; the intervals of the lane's 16 rows are read 8 rows at a time into the registers the LSE had."""
    carry, rec = SET[u & 1], (u + 2) % 6 * META_SZ
    out = [f"LVX_BWD_MASK{u}_%=:"]
    for half in range(2):
        for n in range(4):      # two groups of four interval starts, then their ends
            vg = 2 * half + n % 2
            out.append(f"ds_read_b128 {vr(LSE + 4 * n, 4)}, v{A_META} offset:{rec + 256 + 256 * (n // 2) + 32 * vg}")
        out.append("s_waitcnt lgkmcnt(0)")
        for v in range(8):
            out += [f"v_cmp_ge_i32 s[88:89], v{TOKEN}, v{LSE + v}", f"v_cmp_lt_i32 vcc, v{TOKEN}, v{LSE + 8 + v}",
                    "s_and_b64 vcc, vcc, s[88:89]", f"v_cndmask_b32 v{carry + 8 * half + v}, 0, v{carry + 8 * half + v}, vcc"]
    return out + [f"s_branch LVX_BWD_SEEN{u}_%="]


def p_bias(u):
    """Request of tile i+1's bias in step u, rows clamped to the window's last, and the walk to the tile after it."""
    f = [["s_cmp_eq_u32 s98, 1", "s_cselect_b32 s88, s99, 31"]]
    for n in range(4):
        t = IV + n % 2
        f += [f"v_add_u32 v{t}, {8 * n}, v{BROW}", f"v_min_u32 v{t}, s88, v{t}",
              [f"s_add_i32 m0, s39, {1024 * n}", f"v_mad_u32_u24 v{t}, v{t}, s93, v{BCHUNK}", f"global_load_lds_dwordx4 v{t}, s[96:97]"]]
    f += [["s_add_u32 s96, s96, s94", "s_addc_u32 s97, s97, 0", "s_sub_i32 s98, s98, 1", "s_cmp_lg_u32 s98, 0",
           f"s_cbranch_scc1 LVX_BWD_SAMEBIAS{u}_%=", "s_add_u32 s96, s96, s100", "s_addc_u32 s97, s97, s101", "s_mov_b32 s98, s53",
           f"LVX_BWD_SAMEBIAS{u}_%=:"]]
    return f


def flat(items):
    out = []
    for x in items:
        out += x if isinstance(x, list) else [x]
    return out


def p_step(u, seed):
    """P-wave step i, i % 6 == (u + 3) % 6.  Operands 0..6 were read in the step before."""
    st = Stream(seed)
    e = st.emit
    sl_p = (u + 2) % 6
    par = u & 1                                                  # (i + 1) & 1: P(i-1) hand-over, dS^T(i-3)
    carry, new = SET[u & 1], SET[(u + 1) & 1]
    # tile i+1 has landed: after its loads this wave issued 2 stores, 4 (wave 0: 5) loads and 2 stores
    # (with a bias four loads of that more)
    e(f"s_waitcnt vmcnt({12 if BIAS else 8})")
    e(f"s_waitcnt lgkmcnt({st.n_lds})")
    e("s_barrier")
    for vg in range(4):
        st.lds(f"ds_read_b128 {vr(LSE + 4 * vg, 4)}, v{A_META} offset:{sl_p * META_SZ + vg * 32}", ("lse", vg))
    if MASKED:
        st.lds(f"ds_read_b32 v{IV}, v{A_IV} offset:{sl_p * META_SZ}")
        st.lds(f"ds_read_b32 v{IV + 1}, v{A_IV} offset:{sl_p * META_SZ + 256}", "iv")

    # P(i-1) = exp2(S(i-1) * c - LSE), packed
    valu = []
    for vg in range(4):
        valu.append(lambda vg=vg: st.wait(("lse", vg)))
        for r in range(4 if BIAS else 0):
            v = 4 * vg + r
            valu.append(f"v_fma_f32 v{LSE + v}, v{BV + v}, s95, -v{LSE + v}")
        for r in range(4):
            v = 4 * vg + r
            valu.append(f"v_fma_f32 v{carry + v}, v{carry + v}, s40, {'' if BIAS else '-'}v{LSE + v}")
        for r in range(4):
            valu.append(f"v_exp_f32 v{carry + 4 * vg + r}, v{carry + 4 * vg + r}")
        if vg >= 1 and not MASKED:
            for e2 in range(2):
                v = 4 * (vg - 1) + 2 * e2
                valu.append(f"{CVT} v{PU + v // 2}, v{carry + v}, v{carry + v + 1}")
    if MASKED:
        valu.append(lambda: st.wait("iv"))
        valu.append([f"v_cmp_lt_i32 vcc, s86, v{IV}", f"v_cmp_gt_i32 s[88:89], s87, v{IV + 1}", "s_or_b64 vcc, vcc, s[88:89]",
                     "s_or_b64 vcc, vcc, s[90:91]", f"s_cbranch_vccnz LVX_BWD_MASK{u}_%=", f"LVX_BWD_SEEN{u}_%=:"])
    else:
        valu.append("s_nop 0")
    for v in range(0 if MASKED else 12, 16, 2):
        valu.append(f"{CVT} v{PU + v // 2}, v{carry + v}, v{carry + v + 1}")
    # hand P over to the D-wave
    valu.append(lambda: st.lds(f"ds_write_b128 v{A_PB}, {vr(PU, 4)} offset:{par * PB_SZ}"))
    valu.append(lambda: st.lds(f"ds_write_b128 v{A_PB}, {vr(PU + 4, 4)} offset:{par * PB_SZ + 1024}"))

    # second half: request of tile i+3 and the walk, dS^T(i-3) copy-out.  The loads go first: the wait
    # at the top of a step then leaves the two stores of the step before last in flight as well
    tail = []
    if BIAS:    # behind the loads of tile i's bias the wave issued 4 (wave 0: 5) tile loads and 2 stores
        tail.append("s_waitcnt vmcnt(6)")
        for n in range(0, 16, 2):
            tail.append(lambda n=n: st.lds(f"ds_read2st64_b32 {vr(BV + n, 2)}, v{A_BV} offset0:{n} offset1:{n + 1}", "bias"))
    for n in range(4):
        tail.append(lambda n=n: st.lds(f"ds_read_b64_tr_b16 {vr(CPD + 2 * n, 2)}, v{A_CP[n % 2]} offset:{par * DST_SZ + 1024 * (n // 2)}", f"cp{n}"))
    ws_old = 66 + 2 * (u % 6)          # workspace address of tile i-3 (tile i+3 takes its place below)
    fetch = p_fetch(u, 3)
    if u == 5:      # the last step of the last trip requests nothing: the steps after the loop do
        fetch = [["s_cmp_eq_u32 s64, 1", "s_cbranch_scc1 LVX_BWD_NOFETCH_%="] + flat(fetch) + ["LVX_BWD_NOFETCH_%=:"]]
    # the stores read the workspace address of tile i-3 before the walk overwrites it: keep a copy
    if BIAS:
        tail += [lambda: st.wait("bias")] + p_bias(u)
    tail += [f"s_mov_b64 s[78:79], {sr(ws_old, 2)}"] + fetch + [lambda: st.wait("cp3")]
    tail.append(["s_cmp_eq_u32 s92, 0", f"s_cbranch_scc1 LVX_BWD_KEEP{u}_%=", *p_store(" nt"), f"LVX_BWD_STORED{u}_%=:"])

    mf = []
    for k in range(NOP):
        def m(k=k):
            st.wait(("op", u, k))
            slot = STG + 4 * (k % NSLOT)
            if k < NKK:
                c = "0" if k == 0 else vr(new, 16)
                e(f"{MFMA} {vr(new, 16)}, {vr(slot, 4)}, {vr(BREG + 4 * k, 4)}, {c}")
            else:
                j, dt = (k - NKK) // NDT, (k - NKK) % NDT
                e(f"{MFMA} {vr(ACC + 16 * dt, 16)}, {vr(slot, 4)}, {vr(PU + 4 * j, 4)}, {vr(ACC + 16 * dt, 16)}")
            if k + AHEAD < NOP:
                p_read_op(st, u, k + AHEAD)
            else:
                p_read_op(st, (u + 1) % 6, k + AHEAD - NOP)
        mf.append(m)
    side = valu + tail
    nv = sum(len(x) if isinstance(x, list) else 1 for x in valu)
    nt = sum(len(x) if isinstance(x, list) else 1 for x in tail)
    shares = [-(-nv // NKK)] * NKK + [-(-nt // (2 * NDT - 1))] * (2 * NDT)
    spread(st, mf, side, shares)
    return st.out, st.carry_over((u + 1) % 6)


def p_prologue():
    """Before the first trip: the operands the first step expects to have been read, and tile i+2."""
    st = Stream()
    st.emit("s_waitcnt vmcnt(0)")
    st.emit("s_waitcnt lgkmcnt(0)")
    st.emit("s_barrier")
    for n in range(AHEAD):
        p_read_op(st, 0, n)
    for y in flat(p_fetch(0, 2)):
        st.emit(y)
    st.emit("s_waitcnt lgkmcnt(0)")     # the first step counts on no more in flight than a step leaves
    return st.out


def d_read_op(st, u, n):
    """LDS read of operand n of D-wave step u: dO rows of tile i-1, then Q^T of tile i-2."""
    sl_p, sl_pp = (u + 2) % 6, (u + 1) % 6
    slot = STG + 4 * (n % NSLOT)
    if n < NKK:
        st.lds(f"ds_read_b128 {vr(slot, 4)}, v{RA + n} offset:{sl_p * TILE_B}", ("op", u, n))
    else:
        j, dt = (n - NKK) // NDT, (n - NKK) % NDT
        off = sl_pp * TILE_B + j * 4096
        st.lds(f"ds_read_b64_tr_b16 {vr(slot, 2)}, v{TA + 2 * dt} offset:{off}")
        st.lds(f"ds_read_b64_tr_b16 {vr(slot + 2, 2)}, v{TA + 2 * dt + 1} offset:{off}", ("op", u, n))


def d_step(u, seed):
    """D-wave step i, i % 6 == (u + 3) % 6.  Operands 0..6 were read in the step before."""
    st = Stream(seed)
    e = st.emit
    sl_pp = (u + 1) % 6                        # buffer of tile i-2 (Q^T, metadata)
    par = (u + 1) & 1                          # i & 1: P(i-2) hand-over, dS^T(i-2) staging
    carry, new = SET[u & 1], SET[(u + 1) & 1]
    e(f"s_waitcnt lgkmcnt({st.n_lds})")
    e("s_barrier")
    st.lds(f"ds_read_b128 {vr(PU, 4)}, v{A_PB} offset:{par * PB_SZ}", ("pu", 0))
    st.lds(f"ds_read_b128 {vr(PU + 4, 4)}, v{A_PB} offset:{par * PB_SZ + 1024}", ("pu", 1))
    for q in range(4):
        st.lds(f"ds_read_b128 {vr(DELTA + 4 * q, 4)}, v{A_META} offset:{sl_pp * META_SZ + 128 + q * 32}", ("dl", q))

    # scale * dS(i-2) = P(i-2) * (dP(i-2) * scale - delta * scale), packed
    valu = []
    t = [TMP, TMP + 1, TMP + 2, TMP + 3]
    for q in range(4):          # registers 4q .. 4q+3 of the dP set; P pairs PU[2q], PU[2q+1]
        valu.append(lambda q=q: st.wait(("dl", q)))      # the P reads were issued before the delta reads
        for r in range(4):
            v = 4 * q + r
            valu.append(f"v_fma_f32 v{carry + v}, v{carry + v}, s40, -v{DELTA + v}")
        if F16:     # a half of the packed P times the fp32 value, in one instruction
            for r in range(4):
                v = 4 * q + r
                valu.append(f"v_fma_mix_f32 v{carry + v}, v{PU + 2 * q + r // 2}, v{carry + v}, 0 op_sel:[{r % 2},0,0] op_sel_hi:[1,0,0]")
        else:
            valu.append(f"v_lshlrev_b32 v{t[0]}, 16, v{PU + 2 * q}")
            valu.append(f"v_and_b32 v{t[1]}, 0xffff0000, v{PU + 2 * q}")
            valu.append(f"v_lshlrev_b32 v{t[2]}, 16, v{PU + 2 * q + 1}")
            valu.append(f"v_and_b32 v{t[3]}, 0xffff0000, v{PU + 2 * q + 1}")
            for r in range(4):
                v = 4 * q + r
                valu.append(f"v_mul_f32 v{carry + v}, v{t[r]}, v{carry + v}")
        valu.append(f"{CVT} v{DSU + 2 * q}, v{carry + 4 * q}, v{carry + 4 * q + 1}")
        valu.append(f"{CVT} v{DSU + 2 * q + 1}, v{carry + 4 * q + 2}, v{carry + 4 * q + 3}")
    for vg in range(4):
        valu.append(lambda vg=vg: st.lds(f"ds_write_b64 v{A_DS[vg]}, {vr(DSU + 2 * vg, 2)} offset:{par * DST_SZ}"))

    mf = []
    for k in range(NOP):
        def m(k=k):
            st.wait(("op", u, k))
            slot = STG + 4 * (k % NSLOT)
            if k < NKK:
                c = "0" if k == 0 else vr(new, 16)
                e(f"{MFMA} {vr(new, 16)}, {vr(slot, 4)}, {vr(BREG + 4 * k, 4)}, {c}")
            else:
                j, dt = (k - NKK) // NDT, (k - NKK) % NDT
                e(f"{MFMA} {vr(ACC + 16 * dt, 16)}, {vr(slot, 4)}, {vr(DSU + 4 * j, 4)}, {vr(ACC + 16 * dt, 16)}")
            if k + AHEAD < NOP:
                d_read_op(st, u, k + AHEAD)
            else:
                d_read_op(st, (u + 1) % 6, k + AHEAD - NOP)
        mf.append(m)
    shares = [6] * 8 + [4, 4, 4, 2, 2, 2, 0, 0] if DH == 128 else [12] * 4 + [8, 8, 0, 0]
    spread(st, mf, valu, shares)
    return st.out, st.carry_over((u + 1) % 6)


def d_prologue():
    st = Stream()
    st.emit("s_waitcnt lgkmcnt(0)")
    st.emit("s_barrier")
    for n in range(AHEAD):
        d_read_op(st, 0, n)
    st.emit("s_waitcnt lgkmcnt(0)")     # the first step counts on no more in flight than a step leaves
    return st.out


def check(ins):
    """Hazard lint (conservative): distance in issue slots, an s_nop N counting N + 1."""
    def regs(tok):
        tok = tok.strip().lstrip("-")
        m = re.match(r"v\[(\d+):(\d+)\]$", tok)
        if m:
            return set(range(int(m.group(1)), int(m.group(2)) + 1))
        m = re.match(r"v(\d+)$", tok)
        return {int(m.group(1))} if m else set()
    hist = []
    for line in ins:
        if line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        toks = [t.split(" offset")[0] for t in rest.split(",")] if rest else []
        weight = int(rest) + 1 if op == "s_nop" else 1
        wr, rd, kind = set(), set(), "other"
        if op.startswith("v_mfma"):
            kind, wr = "mfma", regs(toks[0])
            rd = regs(toks[1]) | regs(toks[2]) | regs(toks[3])
        elif op.startswith("v_"):
            kind = "trans" if op.startswith("v_exp") else "valu"
            wr = regs(toks[0])
            rd = set().union(*[regs(x) for x in toks[1:]]) if len(toks) > 1 else set()
        elif op.startswith("ds_read"):
            kind, wr, rd = "lds", regs(toks[0]), regs(toks[1])
        elif op.startswith("ds_write"):
            kind, rd = "lds", regs(toks[0]) | regs(toks[1])
        elif op.startswith("global_store"):
            kind, rd = "vmem", regs(toks[0]) | regs(toks[1])
        elif op.startswith("global_load_lds"):
            kind, rd = "vmem", regs(toks[0])
            if hist and hist[-1][0] == "m0":
                raise SystemExit(f"hazard: {line} right behind the write of M0")
        elif toks and toks[0] == "m0":
            kind = "m0"
        dist = 0
        for pk, pw, pwt in reversed(hist):
            if pk == "mfma" and kind != "mfma" and (pw & (rd | wr)) and dist < 14:
                raise SystemExit(f"hazard: {line} touches an MFMA result after {dist} slots")
            if pk in ("valu", "trans") and kind == "mfma" and (pw & rd) and dist < 3:
                raise SystemExit(f"hazard: {line} reads a VALU result after {dist} slots")
            if pk == "trans" and kind in ("valu", "trans") and (pw & rd) and dist < 2:
                raise SystemExit(f"hazard: {line} reads a transcendental result after {dist} slots")
            dist += pwt
            if dist > 40:
                break
        hist.append((kind, wr, weight))


def main():
    step = p_step if ROLE == "p" else d_step
    # what step 5 leaves to step 0 of the next trip: every step issues the same LDS operations in the
    # same order, so a dry run of one step tells
    _, seed = step(5, {"n": AHEAD, "tag": {("op", 5, k): k + 1 for k in range(AHEAD)}})
    body = []
    for u in range(6):
        ins, left = step(u, seed)
        assert u == 5 or left == {"n": seed["n"], "tag": {("op", u + 1, t[2]): p for t, p in seed["tag"].items()}}, (left, seed)
        seed = left
        body += [x for x in ins if x is not None]
    check(body + body)
    cnt = "s64"
    prologue = p_prologue() if ROLE == "p" else d_prologue()
    check(prologue)
    lines = prologue + ["LVX_BWD_LOOP_%=:"] + body + [f"s_sub_i32 {cnt}, {cnt}, 1", f"s_cmp_lg_u32 {cnt}, 0", "s_cbranch_scc1 LVX_BWD_LOOP_%=",
                                           "s_waitcnt lgkmcnt(0)", "s_nop 15", "s_nop 3"]
    if ROLE == "p":
        lines += ["s_branch LVX_BWD_END_%="] + p_ragged(0, 2)
        for u in range(6):
            lines += p_ragged(u, 3) + p_keep(u) + (p_mask(u) if MASKED else [])
        lines.append("LVX_BWD_END_%=:")
    print("// generated by gen_bwd_loop.py - do not edit")
    for l in lines:
        print(f'"{l}\\n"')


main()

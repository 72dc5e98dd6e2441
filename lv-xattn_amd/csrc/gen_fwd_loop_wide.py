"""Writes the key-tile loop of the forward kernel whose waves own TWO blocks of 32 text rows
(lvx_fwd.hip, fwd_wide_kernel), for one element type and head dimension:

    python gen_fwd_loop_wide.py bf16|f16 128|64 [bias] > lvx_fwd_loop_wide_<type>_<dim>[_bias].inc

The statement runs ALL key tiles of a work-group, one or more.  Per key tile t it issues in program
order the MFMAs of S(t+1) = K(t+1) Q^T and of O += V(t)^T P(t), and between any two of them a few
of the tile's other instructions: the exponentials of tile t, the row maximum of tile t+1, the LDS
operand reads and the global -> LDS loads of K(t+2) and V(t+1).  Every K or V operand read from LDS
feeds two MFMAs, one per row block.  The wave has the SIMD to itself (512 registers): the O^T
accumulators and Q^T live in accumulation registers, which only MFMAs touch (the rare rescale of O
goes through a few VGPRs).

What only some tiles need sits behind the loop as out-of-line blocks the stream tests for with a
scalar compare: the move of a row's reference maximum and the rescale of O, the element mask of a
tile that some row of the work-group does not see in full, and the clamp of the load addresses to
the last row of the key range when the next tile to be requested is the last.

With a dense bias the scores of tile t+1 become S * c + bias * log2(e) before their row maximum is taken, and c is 1 elsewhere.
(S * scale + bias would be an instruction less, but where a row sees nothing above -1e9 its exponents, log2(e) * (x - max) by
one multiply-add, would be as far off as that product's rounding.)  The wave's 64 rows x 64 keys of fp32 come through an LDS tile of its own, 4 rows (1 KiB and 16 bytes of
padding) to a load: a lane's 16 bytes of a key group are then a read without bank conflicts, and loads cover whole cache lines.
There is one such tile: it is read while O += V(t)^T P(t), and refilled from there (BIAS_LATE loads) on into the S phase of the
next tile, in front of that tile's K and V, so that counts of loads in flight tell all of them apart.

Register map (must match the constraints of the asm statement in lvx_fwd.hip), b = row block:
  at entry: v[128 + 2 b : 129 + 2 b] this lane's address in the Q row of block b
  at exit : v[64 b :] O^T of block b, 16 registers per 32 values of d
  inside  : a[64 b :] O^T, a[128 + 32 b :] Q^T
            v[64 b : 64 b + 31] scores set A, v[64 b + 32 : 64 b + 63] scores set B
            v[128 + 16 b : 143 + 16 b] P^T   v[160:199] ten operand slots
  v[200:207] K read addresses (per k-step)   v[208:215] V read addresses (d tile x half)
  v[216:219] / v[220:223] global byte offsets of this wave's pieces of the next K / V tile (at entry: the first)
  v224 what of such an offset is not row * stride   v225+b first visible key - 4 * (lane / 32)
  v227+b visible keys   v229+b m   v231+b l   v233+b alpha   v235+b -m*c   v237+b .. v243+b scratch
  s40 c = scale*log2(e)   s41 -inf   s42 8.0   s[44:45] next K tile   s[46:47] next V tile
  s48 / s49 bytes per K / V tile   s50 LDS address of this wave's part of buffer 0
  s51 tiles after the current one   s57 / s62 tiles after the next K / V tile
  s64 / s65 byte offset of the last row of the key range in its tile (K / V)
  s66 first key of the tile whose scores are formed   s67, s68 no row masks anything in the tiles
  with (s66 - s67) <= s68, unsigned   s[52:53], s[60:61], s[70:71], s56 scratch
  s[54:55], s[58:59] rows whose reference moved in the tile before
  bias: v245 scratch   v246 byte offset of this lane's piece of the next load from the tile's first element
        v[248:251] at entry: read addresses of key groups 0, 16, 32, 48 (a[192:195] inside)
        v[248:255], v[238:241] three read slots   s[72:75] buffer of the next tile, from its first element to the tensor's last
        s76 bytes of 4 rows   s77 LDS address of the wave's tile   s78 scale*log2(e)   s80 log2(e)   s79 tiles after the next bias tile
"""
import os
import re
import sys

# experiment switches (comma separated in LVX_GEN_OPTS); none is set in a normal build
OPTS = dict((o.split("=") + ["1"])[:2] for o in os.environ.get("LVX_GEN_OPTS", "").split(",") if o)
F16 = len(sys.argv) > 1 and sys.argv[1] == "f16"
DH = int(sys.argv[2]) if len(sys.argv) > 2 else 128
BIAS = len(sys.argv) > 3 and sys.argv[3] == "bias"
MFMA = "v_mfma_f32_32x32x16_f16" if F16 else "v_mfma_f32_32x32x16_bf16"
CVT = "v_cvt_pk_f16_f32" if F16 else "v_cvt_pk_bf16_f32"

NKK, NDT = DH // 16, DH // 32       # k-steps of S, 32-wide blocks of O^T
NS, NV = 2 * NKK, 4 * NDT           # operands of the S phase (k-step x key half) and of the V phase
NLD = DH // 32                      # 1 KiB pieces of a tile per wave
ROWB = 2 * DH                       # bytes per row of a tile in LDS
TILE = 64 * ROWB
NB = 2
SC = [[0, 32], [64, 96]]            # score sets [block][set]
PB = [128, 144]
STG, KA, VA, DOK, DOV, LDC = 160, 200, 208, 216, 220, 224
ME, ML = [225, 226], [227, 228]
MI, LI, AL = [229, 230], [231, 232], [233, 234]
NMC = [235, 236]
MX, T0, T1, RS1 = [237, 238], [239, 240], [241, 242], [243, 244]
AACC, AQ = [0, 64], [128, 160]
BADDR, BOFF, BREAD, BSLOT = 245, 246, 192, [248, 252, 238]
BLOCKB = 1040                       # bytes of four rows of bias in LDS
BIAS_LOADS, BIAS_LATE = 16, int(OPTS.get("blate", 8))       # of a tile; of them, in the tile that reads the one before
RMASK = ["s[54:55]", "s[58:59]"]
CMASK = ["s[52:53]", "s[60:61]"]
NSLOT, AHEAD, WBATCH = 10, int(OPTS.get("ahead", 8)), int(OPTS.get("wbatch", 2))
# VALU instructions behind an MFMA of the S / V phase: with heads of 64 the same softmax has half as many
TAKE_S, TAKE_V = (int(OPTS.get("s1", 5 if BIAS else 4)), int(OPTS.get("s2", 7 if BIAS else 5))) if DH == 128 else \
    (int(OPTS.get("s1", 9 if BIAS else 8)), int(OPTS.get("s2", 14 if BIAS else 10)))


def vr(base, n=1):
    return f"v{base}" if n == 1 else f"v[{base}:{base + n - 1}]"


def ar(base, n=1):
    return f"a{base}" if n == 1 else f"a[{base}:{base + n - 1}]"


class Stream:
    """Instruction list with a model of the in-order LDS return queue for s_waitcnt lgkmcnt."""

    def __init__(self):
        self.out = []
        self.lds_issued = 0
        self.ready_after = {}   # operand id -> number of LDS reads issued when its last read was issued

    def emit(self, s):
        if callable(s):
            s()
            return
        if isinstance(s, list):     # instructions that must stay together
            for x in s:
                self.emit(x)
            return
        if "nodma" in OPTS and (s.startswith("global_load_lds") or s.startswith("s_add_i32 m0")):
            return
        if "novalu" in OPTS and s.startswith("v_") and not s.startswith("v_mfma") and not s.startswith("v_acc"):
            return
        self.out.append(s)

    def lds_read(self, text, op):
        if "nolds" not in OPTS:
            self.out.append(text)
        self.lds_issued += 1
        self.ready_after[op] = self.lds_issued

    def wait_op(self, op):
        n = self.lds_issued - self.ready_after[op]
        self.out.append(f"s_waitcnt lgkmcnt({min(n, 15)})")


def exp_group(b, cur, j, nmc, first):
    """P^T k-step j of block b from its score set cur: registers 8j..8j+7 of s0 (j < 2) or s1.
    Exponentials and their consumers are kept at least two instructions apart."""
    base = SC[b][cur] + (16 if j >= 2 else 0) + 8 * (j & 1)
    ins = []
    pend = []
    for e in range(4):
        r0, r1 = base + 2 * e, base + 2 * e + 1
        ins.append(f"v_fma_f32 v{r0}, v{r0}, s40, v{nmc}")
        ins.append(f"v_fma_f32 v{r1}, v{r1}, s40, v{nmc}")
        ins.append(f"v_exp_f32 v{r0}, v{r0}")
        ins.append(f"v_exp_f32 v{r1}, v{r1}")
        ins += pend
        pend = []
        if first and e == 0:
            pend.append(f"v_add_f32 v{RS1[b]}, v{r0}, v{r1}")
        else:
            pend.append(f"v_add_f32 v{LI[b]}, v{LI[b]}, v{r0}")
            pend.append(f"v_add_f32 v{RS1[b]}, v{RS1[b]}, v{r1}")
        pend.append(f"{CVT} v{PB[b] + 4 * j + e}, v{r0}, v{r1}")
    ins.append("s_nop 0")
    ins += pend
    return ins


SLOW = []       # out-of-line code
N_SLOW = [0]


def new_label():
    N_SLOW[0] += 1
    return N_SLOW[0]


def mask_test(nxt):
    """Is the next tile one that some row does not see in full?  Then (out of line) its scores at keys a
    lane's row does not see become -inf, for both row blocks."""
    n = new_label()
    out = [f"LVX_FWDW_MASK{n}_%=:", f"v_mov_b32 v{T1[1]}, s41"]
    pairs = ["s[52:53]", "s[60:61]", "s[70:71]", "vcc"]
    for b in range(NB):
        base = T0[b]
        tmp = [MX[0], MX[1], T1[0], T0[1 - b]]
        out.append(f"v_sub_u32 v{base}, s66, v{ME[b]}")
        for q in range(8):                              # scores 4 q .. 4 q + 3
            regs = [SC[b][nxt] + 4 * q + i for i in range(4)]
            keys = [32 * (q // 4) + 8 * (q % 4) + i for i in range(4)]
            for i in range(4):
                out.append(f"v_add_u32 v{tmp[i]}, {keys[i]}, v{base}")
            for i in range(4):
                out.append(f"v_cmp_lt_u32 {pairs[i]}, v{tmp[i]}, v{ML[b]}")
            out.append("s_nop 1")
            for i in range(4):
                out.append(f"v_cndmask_b32 v{regs[i]}, v{T1[1]}, v{regs[i]}, {pairs[i]}")
    out += ["s_nop 1", f"s_branch LVX_FWDW_MASKED{n}_%="]
    SLOW.extend(out)
    return [["s_sub_u32 s56, s66, s67", "s_cmp_gt_u32 s56, s68", f"s_cbranch_scc1 LVX_FWDW_MASK{n}_%=",
             f"LVX_FWDW_MASKED{n}_%=:"]]


def next_max(b, nxt):
    """Row maximum of the next tile's scores of block b and the test whether any row's reference
    maximum has to move (its maximum grew by more than 2^8 since the reference was set, or there was
    none).  The move itself - alpha, the new reference and -m*c - is rare and sits behind the loop."""
    s0, s1 = SC[b][nxt], SC[b][nxt] + 16
    mx, t0, t1, mi, al, nmc = MX[b], T0[b], T1[b], MI[b], AL[b], NMC[b]
    ins = [f"v_max3_f32 v{mx}, v{s0}, v{s1}, v{s0 + 1}"]
    for v in range(2, 16):
        ins.append(f"v_max3_f32 v{mx}, v{mx}, v{s1 + v - 1}, v{s0 + v}")
    ins.append(f"v_max_f32 v{mx}, v{mx}, v{s1 + 15}")
    n = new_label()
    ins += [
        f"v_mov_b32 v{t0}, v{mx}",
        "s_nop 1",
        f"v_permlane32_swap_b32 v{mx}, v{t0}",
        "s_nop 1",
        f"v_max3_f32 v{mx}, v{mx}, v{t0}, v{mi}",
        # candidate reference mx*c against the current m*c: move when the difference exceeds 8 (or is not
        # a number: no reference yet) and mx is finite
        f"v_mul_f32 v{t0}, s40, v{mx}",
        f"v_fma_f32 v{t0}, -s40, v{mi}, v{t0}",
        f"v_cmp_neq_f32 vcc, s41, v{mx}",
        f"v_cmp_nge_f32 {CMASK[b]}, s42, v{t0}",
        [f"s_and_b64 {RMASK[b]}, vcc, {CMASK[b]}",
         f"s_cbranch_scc1 LVX_FWDW_MOVE{n}_%=",
         f"LVX_FWDW_MOVED{n}_%=:"],
    ]
    SLOW.extend([
        f"LVX_FWDW_MOVE{n}_%=:",
        f"v_mul_f32 v{t0}, s40, v{mx}",
        f"v_fma_f32 v{t1}, s40, v{mi}, -v{t0}",
        f"v_exp_f32 v{t1}, v{t1}",
        "s_nop 1",
        f"v_cndmask_b32 v{al}, 1.0, v{t1}, {RMASK[b]}",
        f"v_cndmask_b32 v{mi}, v{mi}, v{mx}, {RMASK[b]}",
        "s_nop 0",
        f"v_mul_f32 v{nmc}, v{mi}, -s40",
        f"v_cmp_neq_f32 vcc, s41, v{mi}",
        "s_nop 1",
        f"v_cndmask_b32 v{nmc}, 0, v{nmc}, vcc",
        f"s_branch LVX_FWDW_MOVED{n}_%=",
    ])
    return ins


def rescale(b, tag, e):
    """O^T and l of block b times alpha, for the rare tile in which some row's reference maximum moved
    (behind the loop, like the move itself).  The accumulators are out of reach of the VALU: sixteen at
    a time travel through the operand slots, which hold nothing at the top of a tile."""
    e([f"s_cmp_lg_u64 {RMASK[b]}, 0", f"s_cbranch_scc1 LVX_FWDW_RESC{tag}{b}_%=", f"LVX_FWDW_RESCD{tag}{b}_%=:"])
    out = [f"LVX_FWDW_RESC{tag}{b}_%=:", "s_nop 15", "s_nop 3", f"v_mul_f32 v{LI[b]}, v{LI[b]}, v{AL[b]}"]
    for c in range(NDT):
        for r in range(16):
            out.append(f"v_accvgpr_read_b32 v{STG + r}, a{AACC[b] + 16 * c + r}")
        for r in range(16):
            out.append(f"v_mul_f32 v{STG + r}, v{AL[b]}, v{STG + r}")
        for r in range(16):
            out.append(f"v_accvgpr_write_b32 a{AACC[b] + 16 * c + r}, v{STG + r}")
    out += ["s_nop 3", f"s_branch LVX_FWDW_RESCD{tag}{b}_%="]
    SLOW.extend(out)


def advance(left, lo, hi, stride, offs, limit):
    """The source of the next K (V) tile moves on unless it stands at the last tile; when it gets there
    the row part of the offsets is cut to the last row of the key range (out of line)."""
    n = new_label()
    SLOW.append(f"LVX_FWDW_LAST{n}_%=:")
    for j in range(NLD):
        SLOW.extend([f"v_sub_u32 v{MX[0]}, v{offs + j}, v{LDC}", f"v_min_u32 v{MX[0]}, {limit}, v{MX[0]}",
                     f"v_add_u32 v{offs + j}, v{MX[0]}, v{LDC}"])
    SLOW.append(f"s_branch LVX_FWDW_STAY{n}_%=")
    return [f"s_cmp_eq_u32 {left}, 0", f"s_cbranch_scc1 LVX_FWDW_STAY{n}_%=",
            f"s_add_u32 {lo}, {lo}, {stride}", f"s_addc_u32 {hi}, {hi}, 0",
            f"s_sub_u32 {left}, {left}, 1", f"s_cmp_eq_u32 {left}, 0", f"s_cbranch_scc1 LVX_FWDW_LAST{n}_%=",
            f"LVX_FWDW_STAY{n}_%=:"]


def bias_advance():
    """The source of the next bias tile moves on unless it stands at the last tile."""
    n = new_label()
    return [["s_cmp_eq_u32 s79, 0", f"s_cbranch_scc1 LVX_FWDW_BSTAY{n}_%=", "s_add_u32 s72, s72, 256", "s_addc_u32 s73, s73, 0",
             "s_sub_u32 s74, s74, 256", "s_sub_u32 s79, s79, 1", f"LVX_FWDW_BSTAY{n}_%=:"]]


def bias_request(j):
    """The j-th load of the bias tile that the source stands at: rows 4 j .. 4 j + 3."""
    out = [f"s_add_i32 m0, s77, {j * BLOCKB}", "s_nop 0", f"buffer_load_dwordx4 v{BOFF}, s[72:75], 0 offen lds"]
    if j < BIAS_LOADS - 1:
        return [out + [f"v_add_u32 v{BOFF}, s76, v{BOFF}"]]
    return [out + [f"s_mul_i32 s56, s76, {BIAS_LOADS - 1}", f"v_subrev_u32 v{BOFF}, s56, v{BOFF}"]]


def bias_scores(nxt, st, behind):
    """The next tile's scores times scale, plus its bias.  behind: loads in flight behind the bias's last."""
    groups = [(m, b, x) for m in range(4) for b in range(NB) for x in range(2)]      # keys 16 m + 8 x + 4 (lane / 32) ..

    def read(i):
        m, b, x = groups[i]
        if b == 0 and x == 0:
            st.emit(f"v_accvgpr_read_b32 v{BADDR}, a{BREAD + m}")
        st.lds_read(f"ds_read_b128 {vr(BSLOT[i % 3], 4)}, v{BADDR} offset:{8 * BLOCKB * b + 32 * x}", ("bias", i))

    out = [f"s_waitcnt vmcnt({behind})"] + [lambda i=i: read(i) for i in range(3)]
    for i, (m, b, x) in enumerate(groups):
        out.append(lambda i=i: st.wait_op(("bias", i)))
        for r in range(4):
            out.append(f"v_mul_f32 v{BSLOT[i % 3] + r}, s80, v{BSLOT[i % 3] + r}")
        for r in range(4):
            v = SC[b][nxt] + 16 * (m // 2) + 8 * (m % 2) + 4 * x + r
            out.append(f"v_fma_f32 v{v}, v{v}, s78, v{BSLOT[i % 3] + r}")
        if i + 3 < len(groups):
            out.append(lambda i=i: read(i + 3))
    return out


def request(offs, base, lds, between):
    """This wave's pieces of a tile, into the buffer at byte `lds` of the tile buffers.  A load to LDS needs a wait
    state behind the write of M0: an instruction taken from `between`."""
    out = []
    for j in range(NLD):
        out += [f"s_add_i32 m0, s50, {lds + j * 4096}", between.pop(0), f"global_load_lds_dwordx4 v{offs + j}, {base}"]
    return out


def tile(par, do_cur=True, do_next=True, do_dma=True, top=True):
    """One key tile t of the pipelined loop (par = t & 1 relative to the first tile).
    do_cur : P(t) from the current scores, O += V(t)^T P(t)
    do_next: S(t+1) = K(t+1) Q^T into the other score set, its row maximum and reference move
    do_dma : request K(t+2) and V(t+1)"""
    cur, nxt = par, par ^ 1
    st = Stream()
    e = st.emit
    tag = f"{par}{int(do_cur)}{int(do_next)}"
    if top:
        # K(t+1) and V(t) have landed; nobody reads K(t) / V(t-1) any more
        e(f"s_waitcnt vmcnt({BIAS_LATE if BIAS and do_next else 0})")
        e("s_barrier")
        if do_next:
            e("s_add_u32 s66, s66, 64")
    if do_cur:
        for b in range(NB):
            rescale(b, tag, e)

    # operand n: below NS = K (k-step n/2, key half n%2) from buffer par^1; above = V (k-step j, d tile dt) from buffer par
    ops = (list(range(NS)) if do_next else []) + (list(range(NS, NS + NV)) if do_cur else [])

    def read_op(n):
        slot = STG + 4 * (n % NSLOT)
        if n < NS:
            kk, half = n // 2, n % 2
            st.lds_read(f"ds_read_b128 {vr(slot, 4)}, v{KA + kk} offset:{(par ^ 1) * 2 * TILE + half * 32 * ROWB}", n)
        else:
            j, dt = (n - NS) // NDT, (n - NS) % NDT
            off = par * 2 * TILE + j * 16 * ROWB
            st.lds_read(f"ds_read_b64_tr_b16 {vr(slot, 2)}, v{VA + 2 * dt} offset:{off}", n)
            st.lds_read(f"ds_read_b64_tr_b16 {vr(slot + 2, 2)}, v{VA + 2 * dt + 1} offset:{off}", n)

    for n in ops[:AHEAD]:
        read_op(n)

    # VALU work of the tile in dependency order; group_end[(b, j)] = how many of them must have been
    # emitted before the MFMAs that read P^T k-step j of block b
    valu, group_end, first_max = [], {}, 10 ** 9
    n_pre = 0
    if do_cur:
        for j in range(4):
            for b in range(NB):
                valu += exp_group(b, cur, j, NMC[b], j == 0)
                group_end[(b, j)] = len(valu)
            if j == 0:
                n_pre = len(valu)       # one group per block before the first MFMA covers the K read latency
            if j == 1 and not do_next:
                n_pre = len(valu)       # without an S phase the first two P operands have to be there anyway
        for b in range(NB):
            valu.append(f"v_add_f32 v{LI[b]}, v{LI[b]}, v{RS1[b]}")
    if do_next:
        first_max = len(valu)
        if BIAS:
            valu += bias_scores(nxt, st, 2 * NLD)
            valu += bias_advance()
        valu += mask_test(nxt)
        rest = [x for b in range(NB) for x in next_max(b, nxt)]
        if BIAS:        # its refill begins among them
            gap = len(rest) // BIAS_LATE
            for j in reversed(range(BIAS_LATE)):
                rest.insert(j * gap, bias_request(j)[0])
        valu += rest
    for s in valu[:n_pre]:
        e(s)
    pos = n_pre
    # global -> LDS loads: K(t+2) into K buffer par, V(t+1) into V buffer par^1
    dma = []
    if do_dma:
        for j in range(NLD):
            dma.append((f"s_add_i32 m0, s50, {par * 2 * TILE + j * 4096}", f"global_load_lds_dwordx4 v{DOK + j}, s[44:45]"))
        for j in range(NLD):
            dma.append((f"s_add_i32 m0, s50, {(par ^ 1) * 2 * TILE + TILE + j * 4096}", f"global_load_lds_dwordx4 v{DOV + j}, s[46:47]"))
    early = [bias_request(j)[0] for j in range(BIAS_LATE, BIAS_LOADS)] if BIAS and do_dma else []
    # operands of the S phase behind which a load of K or V goes: every other one, or those the bias has left
    n_early = NS // 4 if BIAS else 0
    at_dma = [k for k in range(NS) if k % 2 == 1] if not BIAS else [n_early + i * (NS - n_early) // (2 * NLD) for i in range(2 * NLD)]
    n_mfma = 0
    last_s = -100       # index of the last S MFMA
    for i, k in enumerate(ops):
        if i % WBATCH == 0:         # one wait covers the operands of the next few MFMA pairs
            st.wait_op(ops[min(i + WBATCH - 1, len(ops) - 1)])
        slot = STG + 4 * (k % NSLOT)
        for b in range(NB):
            if k < NS:
                kk, half = k // 2, k % 2
                d = SC[b][nxt] + 16 * half
                c = "0" if kk == 0 else vr(d, 16)
                e(f"{MFMA} {vr(d, 16)}, {vr(slot, 4)}, {ar(AQ[b] + 4 * kk, 4)}, {c}")
                last_s = n_mfma
            else:
                j, dt = (k - NS) // NDT, (k - NS) % NDT
                assert pos >= group_end[(b, j)], f"P^T k-step {j} of block {b} is not ready at operand {k}"
                a = AACC[b] + 16 * dt
                e(f"{MFMA} {ar(a, 16)}, {vr(slot, 4)}, {vr(PB[b] + 4 * j, 4)}, {ar(a, 16)}")
            n_mfma += 1
            if b == NB - 1:
                x, y = dma[at_dma.index(k)] if dma and k in at_dma else (None, None)
                if k < n_early:
                    for z in early[k * len(early) // n_early:(k + 1) * len(early) // n_early]:
                        e(z)
                if x:
                    e(x)
                if i + AHEAD < len(ops):        # between the write of M0 and the load: its wait state
                    read_op(ops[i + AHEAD])
                if y:
                    e(y)
                if do_dma and k == NS - 1:
                    e(advance("s57", "s44", "s45", "s48", DOK, "s64"))
                    e(advance("s62", "s46", "s47", "s49", DOV, "s65"))
            take = (TAKE_S if k < NS else TAKE_V) if do_next else 7 * 128 // DH
            if i == len(ops) - 1 and b == NB - 1:
                take = len(valu) - pos
            for _ in range(take):
                if pos >= len(valu):
                    break
                # the row maximum reads the scores the S MFMAs wrote: not before the last of them has had
                # its wait states - with the V MFMAs behind it, no earlier than three MFMAs later
                if pos >= first_max and (n_mfma - 1 < last_s + 4 or k < NS):
                    break
                e(valu[pos])
                pos += 1
    if pos < len(valu):     # S phase alone (prologue): the maximum follows the last MFMA
        e("s_nop 15")
        e("s_nop 3")
        for s in valu[pos:]:
            e(s)
    return st.out


def check(ins):
    """Hazard lint of one tile's stream (conservative): distance in instructions, an s_nop N counting N+1."""
    def regs(tok):
        tok = tok.strip().lstrip("-")
        m = re.match(r"([va])\[(\d+):(\d+)\]$", tok)
        if m:
            return set((m.group(1), r) for r in range(int(m.group(2)), int(m.group(3)) + 1))
        m = re.match(r"([va])(\d+)$", tok)
        return {(m.group(1), int(m.group(2)))} if m else set()
    hist = []   # (kind, written regs, weight)
    for line in ins:
        if line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        toks = [t for t in rest.split(",")] if rest else []
        toks = [t.split(" offset")[0] for t in toks]
        weight = 1
        if op == "s_nop":
            weight = int(rest) + 1
        wr, rd = set(), set()
        kind = "other"
        if op.startswith("v_mfma"):
            kind = "mfma"
            wr = regs(toks[0])
            rd = regs(toks[1]) | regs(toks[2]) | regs(toks[3])
        elif op.startswith("v_cmp"):
            kind = "valu"
            rd = set().union(*[regs(t) for t in toks[1:]])
        elif op.startswith("v_permlane"):
            kind = "valu"
            wr = regs(toks[0]) | regs(toks[1])
            rd = wr
        elif op.startswith("v_"):
            kind = "trans" if op.startswith("v_exp") else "valu"
            wr = regs(toks[0])
            rd = set().union(*[regs(t) for t in toks[1:]]) if len(toks) > 1 else set()
        elif op.startswith("ds_read"):
            kind = "lds"
            wr = regs(toks[0])
            rd = regs(toks[1])
        elif op.startswith("global_load_lds") or op.startswith("buffer_load"):
            kind = "vmem"
            rd = regs(toks[0])
            if hist and hist[-1][0] == "m0":
                raise SystemExit(f"hazard: {line} right behind the write of M0")
        elif toks and toks[0] == "m0":
            kind = "m0"
        dist = 0
        for pk, pw, pwt in reversed(hist):
            if pk == "mfma" and kind != "mfma" and (pw & (rd | wr)) and dist < 14:
                raise SystemExit(f"hazard: {line} touches an MFMA result after {dist} wait states")
            if pk in ("valu", "trans") and kind == "mfma" and (pw & rd) and dist < 3:
                raise SystemExit(f"hazard: {line} reads a VALU result after {dist} wait states")
            if pk == "trans" and kind in ("valu", "trans") and (pw & rd) and dist < 2:
                raise SystemExit(f"hazard: {line} reads a transcendental result after {dist} wait states")
            if pk == "valu" and op.startswith("v_permlane") and (pw & rd) and dist < 2:
                raise SystemExit(f"hazard: {line} reads a VALU result after {dist} wait states")
            dist += pwt
            if dist > 40:
                break
        hist.append((kind, wr, weight))


def main():
    # Entry.  What the first scores need is requested first, K(0) and Q^T - Q^T straight into the accumulation
    # registers it lives in - then V(0) and K(1), which the wait leaves in flight.  O^T starts at 0 meanwhile.
    zero = [f"v_accvgpr_write_b32 a{AACC[b] + r}, 0" for b in range(NB) for r in range(16 * NDT)]
    pro = request(DOK, "s[44:45]", 0, zero) + advance("s57", "s44", "s45", "s48", DOK, "s64")
    for b in range(NB):
        for kk in range(NKK):
            pro.append(f"global_load_dwordx4 {ar(AQ[b] + 4 * kk, 4)}, {vr(128 + 2 * b, 2)}, off offset:{32 * kk}")
    if BIAS:
        pro += [f"v_accvgpr_write_b32 a{BREAD + m}, v{248 + m}" for m in range(4)]
        for j in range(BIAS_LOADS):
            pro += bias_request(j)[0]
    pro += request(DOV, "s[46:47]", TILE, zero) + advance("s62", "s46", "s47", "s49", DOV, "s65")
    pro += request(DOK, "s[44:45]", 2 * TILE, zero) + advance("s57", "s44", "s45", "s48", DOK, "s64")
    pro += zero
    for b in range(NB):
        pro += [f"v_mov_b32 v{MI[b]}, s41", f"v_mov_b32 v{LI[b]}, 0", f"v_mov_b32 v{NMC[b]}, 0"]
    pro += [f"s_waitcnt vmcnt({2 * NLD + (BIAS_LOADS if BIAS else 0)})", "s_barrier"]
    # scores of the first tile (from K buffer 0 into score set A: the S phase of an odd tile)
    pro += tile(1, do_cur=False, do_next=True, do_dma=False, top=False)
    # there is nothing to rescale yet
    pro += ["s_mov_b64 s[54:55], 0", "s_mov_b64 s[58:59], 0"]
    t0, t1 = tile(0), tile(1)
    f0, f1 = tile(0, do_next=False, do_dma=False), tile(1, do_next=False, do_dma=False)
    check(pro + t0 + t1 + t0 + f1)
    check(pro + t0 + t1 + f0)
    check(pro + f0)
    lines = pro + ["LVX_FWDW_LOOP_%=:", "s_cmp_eq_u32 s51, 0", "s_cbranch_scc1 LVX_FWDW_FIN0_%="] + t0
    lines += ["s_cmp_eq_u32 s51, 1", "s_cbranch_scc1 LVX_FWDW_FIN1_%="] + t1
    lines += ["s_sub_u32 s51, s51, 2", "s_branch LVX_FWDW_LOOP_%="]
    lines += SLOW
    lines += ["LVX_FWDW_FIN1_%=:"] + f1 + ["s_branch LVX_FWDW_END_%="]
    lines += ["LVX_FWDW_FIN0_%=:"] + f0 + ["LVX_FWDW_END_%=:", "s_nop 15", "s_nop 3"]
    # Exit: O^T comes down.
    for b in range(NB):
        for r in range(16 * NDT):
            lines.append(f"v_accvgpr_read_b32 v{64 * b + r}, a{AACC[b] + r}")
    lines += ["s_nop 3"]
    print("// generated by gen_fwd_loop_wide.py - do not edit")
    for l in lines:
        print(f'"{l}\\n"')


main()

// Cross-attention backward for gfx950 from the saved LSE and delta:
//   P = exp(scale*Q K^T - LSE);  dV = P^T dO;  dP = dO V^T;
//   dS = P * (dP - delta);  dK = scale * dS^T Q;  dQ = scale * dS K.
//
// Mapping.  A work-group owns a block of 128 visual tokens of one kv head and
// streams every text row of the window for every q head of the GQA group past
// it, 32 rows at a time.  It has 8 waves, two per SIMD, in two roles; waves w
// and w+4 share token slice 32w..32w+31 of the block:
//   P-wave  (w)   : S = Q K^T, P = exp2(..), dV^T += dO^T P     K rows + dV^T resident
//   D-wave  (w+4) : dP = dO V^T, dS = P (dP - delta) scale,
//                   dK^T += Q^T dS                              V rows + dK^T resident
// so each wave keeps 64 accumulator registers and 32 operand registers for the
// whole kernel (the sum over the q heads of the group and over all rows never
// leaves the register file) and fits two to a SIMD: while one wave waits for
// LDS or runs its exp2/multiplies, the other feeds the MFMA pipe.  P travels
// from the P-wave to the D-wave as bf16 through LDS (32 bytes per lane), one
// step behind, so the one barrier per step also orders that hand-over.
//
// dQ = scale * dS K sums over ALL tokens, i.e. over every work-group of the kv
// head.  Adding 51 partial tiles per row with fp32 atomics costs more than the
// whole rest of the kernel on this machine (atomic adds sustain about 1.3 TB/s),
// so dQ is not formed here: the D-waves gather scale*dS (bf16) in LDS and the
// group streams it to a workspace in HBM, one contiguous 8 KB tile
// of 128 tokens x 32 rows per step, indexed [b, h, token block, row tile]; dq_kernel
// (launched by the caller right after) contracts it with K.  The tile is turned on its way out of the LDS: it lies as
// [token / 8][row][8 tokens], so that a lane's operand of that contraction is 16 bytes that it loads from memory into its
// registers.  The workspace costs 2 bytes per
// (row, token, head), written once and read once; the caller says when it is large enough for
// streaming stores (ds_stream).
//
// All MFMA are 32x32x16 bf16.  A operands come from LDS.  The Q and dO tiles
// ([32 rows][128] bf16, 8 KiB each) go from global memory straight into LDS
// with global_load_lds_dwordx4, two steps ahead, into rings of six buffers;
// the load writes 64 lanes x 16 bytes contiguously, so rows are not padded:
// the 16-byte chunk c of row r is kept at position c ^ f(r),
// f(r) = ((r & 3) << 2) | ((r >> 2) & 3), which makes both access patterns
// conflict-free on ONE copy of a tile - Q / dO rows by 16-byte reads, Q^T /
// dO^T by the transposing LDS read, the latter addressed in the accumulator's
// row order so that P / dS go from the registers straight into the next MFMA
// as B operands.  Every wave requests all LDS operands of a step before its
// first MFMA, so their latency is paid once per step.
#include <cstddef>
#include <type_traits>

#include "lvx_common.hpp"
#include "lvx_fold.hpp"
#include "lvx_kernels.hpp"

namespace lvx {

namespace {

constexpr int D = 128;
constexpr int BN = 128;       // visual tokens per work-group
constexpr int BM = 32;        // text rows per step
constexpr int NT = 512;       // threads per work-group

// LDS map (uint16 units): a ring of six Q tiles, a ring of six dO tiles (each ring within the 64 KiB an LDS
// instruction's immediate offset reaches from one address register), unpadded; two dS^T tiles; two P
// hand-over buffers
constexpr int TILE_ELEMS = BM * D;             // one Q or dO tile (8 KiB)
constexpr int NQD = 6;
constexpr int DST_ELEMS = BN * BM;             // [token][row], the 16-byte chunk c of a token at c ^ ((token >> 2) & 3)
constexpr int PB_ELEMS = 4 * 2 * 64 * 8;       // P hand-over: [slice][half][lane][16 bytes] as uint16
constexpr int OFF_Q = 0;                       // x NQD
constexpr int OFF_DO = OFF_Q + NQD * TILE_ELEMS; // x NQD
constexpr int OFF_DST = OFF_DO + NQD * TILE_ELEMS; // x2
constexpr int OFF_PB = OFF_DST + 2 * DST_ELEMS;  // x2
constexpr int OFF_BIAS = OFF_PB + 2 * PB_ELEMS;  // masked with a dense bias: four tiles of 32 rows x 32 tokens fp32, one per P-wave
constexpr int BIAS_ELEMS = 4 * 32 * 32 * 2;
constexpr int EPI_ELEMS = 8 * 32 * (D + 4) * 2;     // 8 waves x [32 tokens][128 + 4] floats of the epilogue, in uint16 units
constexpr int smem_elems(bool bias) {
    const int loop = OFF_BIAS + (bias ? BIAS_ELEMS : 0);
    return loop > EPI_ELEMS ? loop : EPI_ELEMS;
}

constexpr uint32_t META_B = 768;   // bytes of a tile's metadata
constexpr float LOG2E = 1.4426950408889634f;

// registers the hand-scheduled loops use besides their operands (see gen_bwd_loop.py)
#define LVX_BWD_LOOP_CLOBBERS "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127", "v128", "v129", "v130", "v131", "v132", "v133", "v134", "v135", "v136", "v137", "v138", "v139", "v140", "v141", "v142", "v143", "v144", "v145", "v146", "v147", "v148", "v149", "v150", "v151", "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159", "v160", "v161", "v162", "v163", "v164", "v165", "v166", "v167", "v168", "v169", "v170", "v171", "v172", "v173", "v174", "v175", "v176", "v177", "v178", "v179", "v180", "v181", "v182", "v183", "v184", "v185", "v186", "v187", "v188", "v189", "v190", "v191", "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199"

// operands of the hand-scheduled loops, one list per role for all element types, head dimensions and masks
#define LVX_BWD_COMMON_OUT "+{v[0:15]}"(acc[0]), "+{v[16:31]}"(acc[1]), "+{v[32:47]}"(acc[2]), "+{v[48:63]}"(acc[3]), \
    "+{v[96:111]}"(carry), "+{s64}"(trips)
#define LVX_BWD_COMMON_IN "{v[64:67]}"(breg[0]), "{v[68:71]}"(breg[1]), "{v[72:75]}"(breg[2]), "{v[76:79]}"(breg[3]), \
    "{v[80:83]}"(breg[4]), "{v[84:87]}"(breg[5]), "{v[88:91]}"(breg[6]), "{v[92:95]}"(breg[7]),                      \
    "{v200}"(ra[0]), "{v201}"(ra[1]), "{v202}"(ra[2]), "{v203}"(ra[3]),                                              \
    "{v204}"(ra[4]), "{v205}"(ra[5]), "{v206}"(ra[6]), "{v207}"(ra[7]),                                              \
    "{v208}"(ta[0]), "{v209}"(ta[1]), "{v210}"(ta[2]), "{v211}"(ta[3]),                                              \
    "{v212}"(ta[4]), "{v213}"(ta[5]), "{v214}"(ta[6]), "{v215}"(ta[7]), "{v216}"(a_pb), "{v217}"(a_meta)
#define LVX_BWD_P_OUT                                                                                                \
    LVX_BWD_COMMON_OUT, "+{s[44:45]}"(qp), "+{s[46:47]}"(dop), "+{s[48:49]}"(mp), "+{s[50:51]}"(wn), "+{s52}"(left), \
      "+{s[66:67]}"(w0), "+{s[68:69]}"(w1), "+{s[70:71]}"(w2), "+{s[72:73]}"(w3), "+{s[74:75]}"(w4), "+{s[76:77]}"(w5), \
      "+{v221}"(g_t[0]), "+{v222}"(g_t[1]), "+{v223}"(g_t[2]), "+{v224}"(g_t[3]), "+{v225}"(g_meta)
#define LVX_BWD_P_IN                                                                                                 \
    LVX_BWD_COMMON_IN, "{v218}"(a_cp0), "{v219}"(a_cp1), "{v220}"(g_cp), "{v232}"(past_iv),                        \
      "{v226}"(past0), "{v227}"(past1), "{v228}"(a_iv), "{v231}"(token), "{s83}"(uniform32(qrow_b)), "{s84}"(uniform32(dorow_b)), \
      "{s40}"(uniform32(c)), "{s41}"(uniform32((uint32_t)BM * qrow_b)), "{s42}"(uniform32((uint32_t)BM * dorow_b)),  \
      "{s53}"(uniform32(n_live)), "{s[54:55]}"(hdq), "{s[56:57]}"(hddo), "{s[60:61]}"(hdws), "{s[80:81]}"(hdm),      \
      "{s62}"(uniform32(lds0 + (uint32_t)slice * 2048u)), "{s63}"(uniform32(meta0 + meta_w)),                        \
      "{s65}"(uniform32(wave < META_WAVES ? 1 : 0)), "{s82}"(uniform32(ragged ? 1 : -1)),                            \
      "{s85}"(uniform32(meta_w ? BM * 4 : 256)), "{s86}"(uniform32(slice_lo)), "{s87}"(uniform32(slice_lo + 32)),     \
      "{s92}"(uniform32(p.ds_stream)),                                                                               \
      "{s[90:91]}"(uniform64(slice_valid ? (int64_t)0 : (int64_t)-1))
#define LVX_BWD_P_CLOBBERS "memory", "vcc", "scc", "m0", "s78", "s79", "s88", "s89", "v229", "v230", LVX_BWD_LOOP_CLOBBERS
#define LVX_BWD_P_OPERANDS : LVX_BWD_P_OUT : LVX_BWD_P_IN : LVX_BWD_P_CLOBBERS
#define LVX_BWD_P_BIAS_OPERANDS                                                                                      \
    : LVX_BWD_P_OUT, "+{v[234:249]}"(bv), "+{s[96:97]}"(bp), "+{s98}"(b_left)                                     \
    : LVX_BWD_P_IN, "{v233}"(a_bias), "{v250}"(b_row), "{v251}"(b_chunk), "{s39}"(uniform32(lds_bias)),               \
      "{s93}"(uniform32(brow_b)), "{s94}"(uniform32((uint32_t)BM * brow_b)), "{s95}"(uniform32(LOG2E)),               \
      "{s99}"(uniform32(ragged ? last : BM - 1)), "{s[100:101]}"(hdb)                                                \
    : LVX_BWD_P_CLOBBERS
#define LVX_BWD_D_OPERANDS                                                                                           \
    : LVX_BWD_COMMON_OUT : LVX_BWD_COMMON_IN, "{v218}"(a_ds[0]), "{v223}"(a_ds[1]), "{v224}"(a_ds[2]), "{v225}"(a_ds[3]), "{s40}"(uniform32(p.scale))                            \
    : "memory", "vcc", "scc", LVX_BWD_LOOP_CLOBBERS, "v219", "v220", "v221", "v222"

// BIAS: a dense fp32 bias joins the exponent, P = exp2(S*c + bias*log2e - LSE*log2e).
// DH: head dimension, 16, 32, 64 or 128.  The LDS tiles keep their 256-byte rows and chunk
// permutation whatever DH is: below 128 only the first DH / 8 chunks of a row hold data (the
// lanes that would load the others repeat a chunk of the same row), and the k-steps of S / dP
// and the 32-wide blocks of dV^T / dK^T past DH do not exist.  With 16 the one block of dV^T /
// dK^T is half real: its upper 16 rows are products with those repeated chunks, never stored.
template <int DH, bool MASKED, bool BIAS, bool F16>
__global__ __launch_bounds__(NT, 1) void bwd_kernel(const BwdParams p) {
    using E = Elt<F16>;
    static_assert(DH == 16 || DH == 32 || DH == 64 || DH == 128, "head dimension");
    constexpr int NKK = DH / 16, NDT = DH >= 32 ? DH / 32 : 1;
    constexpr int META_WAVES = MASKED ? 3 : 1;      // waves that fetch a part of a tile's metadata
    constexpr int SMEM_ELEMS = smem_elems(MASKED && BIAS && DH >= 64);
    __shared__ __attribute__((aligned(1024))) uint16_t smem[SMEM_ELEMS];
    // per-row metadata of a staged tile, one per tile buffer: 8 x 16 bytes each of LSE*log2e and
    // delta*scale; with an interval mask kv_start and kv_end follow, each twice (a load moves 64 lanes)
    __shared__ __attribute__((aligned(256))) u32x4 meta_s4[NQD][META_B / 16];

    // Work-group ids are dealt to the 8 XCDs round-robin.  XCD x takes the token blocks
    // [x * blocks_per_xcd, (x + 1) * blocks_per_xcd) of the list (b, kv head, block), so that the
    // work-groups of a kv head share an L2: first `whole_blocks` of them with one work-group
    // each, then `mid_blocks` with q_splits work-groups each, then the others with q_splits2
    // each - the longer work-groups first.  (A placement hint only: every (block, range) is
    // produced exactly once whatever the hardware does with the ids.)
    fetch_kernargs<offsetof(BwdParams, dq_before)>();
    if ((int)blockIdx.x >= p.own_wg) {
        // Rounds: the slices of dQ of the round before, summed while the last token blocks leave CUs idle (256 rows of 32 heads, 6404
        // tokens: 408 blocks of equal length on 256 CUs); sixteen, forward and backward, 2773 -> 2743 us.
        const uint32_t i = blockIdx.x - p.own_wg;
        cast_t<F16>(p.dq_before, (int64_t)((i & 7) * p.dq_before.blocks_per_xcd + (i >> 3)) * NT + threadIdx.x);
        return;
    }
    const int xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const int blk0 = xcd * p.blocks_per_xcd;
    const int nblk = min(p.blocks_per_xcd, p.n_blocks - blk0);
    const int whole = max(0, min(p.whole_blocks, nblk));
    const int mid = max(0, min(p.mid_blocks, nblk - whole));
    int blk, S = 1;
    uint32_t sp = 0, kblk, b;
    if (MASKED && p.plan) {
        const uint32_t* const e = p.plan + (int64_t)(xcd * p.per_xcd + local) * PLAN_ENTRY;
        const uint32_t what = __builtin_amdgcn_readfirstlane(e[0]);
        if (what == ~0u) return;
        blk = blk0 + (int)(what & 0xffffu);
        S = (int)(what >> 16 & 0xffu);
        sp = what >> 24;
    } else if (local < whole) {
        blk = blk0 + local;
    } else if (local < whole + mid * p.q_splits) {
        S = p.q_splits;
        blk = blk0 + whole + p.by_splits.split(local - whole, sp);
    } else {
        S = p.q_splits2;
        blk = blk0 + whole + mid + p.by_splits2.split(local - whole - mid * p.q_splits, sp);
        if (blk >= blk0 + nblk) return;
    }
    const uint32_t bh = p.by_kv_blocks.split(blk, kblk);
    const uint32_t hk = p.by_B.split(bh, b);        // samples interleaved: ragged samples then share the tail of the launch

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int slice = wave & 3;
    const bool d_role = wave >= 4;

    int kv_len = p.Lkv;
    if (p.kv_len) kv_len = min(p.kv_len[b], p.Lkv);
    const int kvb = kblk * BN;
    const int my_kv = kvb + 32 * slice + l32;
    const bool kv_valid = my_kv < kv_len;
    const int slice_lo = kvb + 32 * slice;              // this wave's 32 tokens
    const bool slice_valid = slice_lo + 32 <= kv_len;   // all of them inside the sample
    const bool tail_block = kvb + BN > kv_len;

    // steps of this work-group: a contiguous range of the (head, row tile) list
    const int n_qtiles = (p.row_end - p.row_begin + BM - 1) / BM;
    // with an interval mask only the listed runs of tiles are visited (kept in scalar
    // registers), and the splits share that shorter walk evenly
    int run_s[4] = {0, 0, 0, 0}, run_n[4] = {n_qtiles, 0, 0, 0};
    int n_live = n_qtiles;
    if (MASKED && p.live_runs) {
        const int32_t* lr = p.live_runs + ((int64_t)b * p.n_kv_blocks + kblk) * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            run_s[i] = __builtin_amdgcn_readfirstlane(lr[2 * i]);
            run_n[i] = __builtin_amdgcn_readfirstlane(lr[2 * i + 1]);
        }
        n_live = run_n[0] + run_n[1] + run_n[2] + run_n[3];
    }
    const int split_steps = S == 1 ? p.G * n_live : (p.G * n_live + S - 1) / S;
    auto sel4 = [](int r, const int (&a)[4]) { return r == 0 ? a[0] : r == 1 ? a[1] : r == 2 ? a[2] : a[3]; };
    const int it_lo = sp * split_steps;
    const int n_iter = (kvb < kv_len) ? max(0, min(split_steps, p.G * n_live - it_lo)) : 0;
    // nothing to visit and nothing to overwrite: done (bf16 outputs, mode 0, still get their zeros)
    // a block that its work-group owns alone is written by it directly, also when others are shared
    const bool alone = p.dkv_mode == 2 && S == 1;
    const int dkv_mode = S > 1 && p.slices ? 3 : alone ? p.whole_mode : p.dkv_mode;
    if (n_iter == 0 && dkv_mode != 0 && dkv_mode != 3) return;

    // ---- resident B operand: this wave's K rows (P-wave) or V rows (D-wave)
    bf16x8 breg[8];     // [NKK .. 8) stay unused when DH < 128
    {
        const uint16_t* base = d_role ? p.v + b * p.vs.b + hk * p.vs.h + (int64_t)my_kv * p.vs.s
                                      : p.k + b * p.ks.b + hk * p.ks.h + (int64_t)my_kv * p.ks.s;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) breg[kk] = as_bf16x8(ldg16(base + (kk < NKK ? kk : 0) * 16 + g * 8, kv_valid));
    }
    // ---- resident accumulator: dV^T (P-wave) or dK^T (D-wave), [128 d][32 tokens]
    f32x16 acc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[dt][v] = 0.f;

    const float c = p.scale_log2e;

    // global -> LDS is the P-waves' job (their step is the shorter one): P-wave w moves
    // rows 8w..8w+7 of the Q tile and of the dO tile as two 1 KiB loads each (4 rows
    // per load); lane i fills position i & 15 of row 4 ch + (i >> 4), ch = 2w, 2w+1.
    const int ld_r = 8 * slice + (lane >> 4);          // first of the two rows, the other is 4 further
    const uint32_t ld_c0 = (uint32_t)(((lane & 15) ^ (((lane >> 4) << 2) | ((2 * slice) & 3))) & (DH / 8 - 1)) * 16u;
    const uint32_t ld_c1 = (uint32_t)(((lane & 15) ^ (((lane >> 4) << 2) | ((2 * slice + 1) & 3))) & (DH / 8 - 1)) * 16u;
    const uint32_t qrow_b = (uint32_t)p.qs.s * 2u, dorow_b = (uint32_t)p.dos.s * 2u;   // bytes per text row
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t meta0 = (uint32_t)(uintptr_t)&meta_s4[0][0];
    // per-lane offsets: transposing operand reads (rows in accumulator order),
    // P hand-over slot, dS^T copy-out (512 chunks of 16 bytes, one per thread)
    // rows: 16 bytes at row * 256 + ((2 kk + g) ^ f(row)) * 16
    const uint32_t row_rd = (uint32_t)(l32 * 256);
    const uint32_t row_h = (uint32_t)((g ^ (((l32 & 3) << 2) | ((l32 >> 2) & 3))) << 4);
    // transposed, rows in accumulator order: first half rows 16 j + 4 g + r, second
    // half 8 rows further down (its f differs in bit 1); add j * 4096
    uint32_t t_rd[4][2];
    {
        const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
        const int low = (2 * u + (t >> 1)) ^ g;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            t_rd[dt][0] = (uint32_t)((4 * g + r) * 256 + (4 * (dt ^ r) + low) * 16 + (t & 1) * 8);
            t_rd[dt][1] = (uint32_t)((4 * g + r + 8) * 256 + (4 * (dt ^ r) + (low ^ 2)) * 16 + (t & 1) * 8);
        }
    }
    const int pb_off = slice * (2 * 64 * 8) + lane * 8;
    // dS^T copy-out, also by the P-waves: two chunks of 8 tokens of row l32 per lane, four tokens from each of two
    // transposing reads.  Writes of 8 bytes (4 rows of a token) and these reads are both conflict-free.  (In rows of 80 bytes,
    // copied out as they lay, 13 % of the kernel's LDS cycles were conflicts.)  A wave takes its own 32 tokens, 8 g .. and
    // 16 + 8 g .. of the slice; with heads of 16, where these stores are what bounds the kernel, 16 of each half of the block, so that the
    // four waves' first stores lie next to each other, 4 KB.  Forward and backward, us, 2 x 16 heads of 16, 1880 rows x 22890
    // tokens 1865 -> 1780 (rows written as they lay 1815), 16, 1888 x 30000 1264 -> 1248 (1208), 16 of 3000 x 16000 999 -> 1002
    // (1042); heads of 32, 2 x 16, 1880 x 22890 would go from 1948 to 1973.
    constexpr int CP = DH >= 32 ? 32 : 16, CP2 = DH >= 32 ? 16 : 64;   // tokens from wave to wave, from the first chunk to the second
    uint32_t cp_rd[2];                 // of the first chunk
    {
        const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
#pragma unroll
        for (int half = 0; half < 2; ++half)
            cp_rd[half] = (uint32_t)((CP * slice + 8 * g + 4 * half + r) * 64 + ((2 * u + (t >> 1)) ^ (2 * g + half)) * 16 + (t & 1) * 8);
    }
    // workspace tile (b, h, token block, row tile): [16 groups of 8 tokens][32 rows][8 tokens], 8 KB, contiguous
    uint16_t* ws_lane = p.ds_ws + (int64_t)kblk * p.ws_ld + (4 * CP * slice + lane) * 8;

    // The walk over (head of the group, 32-row tile): per-head base addresses are
    // re-derived only when the head changes, everything else advances by constants.
    int cur_gi = 0, cur_run = 0, cur_qt = 0, cur_left = 1;    // cur_left: tiles left in the run, this one included
    if (n_iter > 0) {
        int idx = 0;
        if (it_lo > 0) {
            cur_gi = it_lo / n_live;
            idx = it_lo % n_live;
        }
        while (idx >= sel4(cur_run, run_n)) { idx -= sel4(cur_run, run_n); ++cur_run; }
        cur_qt = sel4(cur_run, run_s) + idx;
        cur_left = sel4(cur_run, run_n) - idx;
    }
    const char* q_head = nullptr;      // Q, dO of (b, head)
    const char* do_head = nullptr;
    const float* meta_head = nullptr;  // metadata records of (b, head)
    int64_t ws_head = 0;               // dS^T workspace offset of (b, head), elements
    auto enter_head = [&]() {
        const int h = hk * p.G + cur_gi;
        q_head = reinterpret_cast<const char*>(p.q + b * p.qs.b + h * p.qs.h);
        do_head = reinterpret_cast<const char*>(p.dout + b * p.dos.b + h * p.dos.h);
        meta_head = p.meta + ((int64_t)b * p.Hq + h) * n_qtiles * 64;
        ws_head = ((int64_t)b * p.Hq + h) * p.ws_bh;
    };
    enter_head();

    // Every load is unconditional and goes straight to LDS: rows past the window are
    // clamped to its last row (their LSE record is +inf, so P = 0 and nothing they
    // carry reaches a result).  Wave 0 also fetches the tile's metadata record
    // (32 x LSE*log2e, 32 x delta*scale; 256 bytes) and, with an interval mask, waves
    // 1 and 2 the rows' first and last keys, ahead of their tile loads so that "tile landed" implies both.
    // more scalars than registers (see dma16); the second load of an address finds it settled
    constexpr bool RESTORED = MASKED && BIAS;
    auto prefetch = [&](int buf) {
        const int r0 = p.row_begin + cur_qt * BM;
        if (wave < META_WAVES) {
            const char* src = reinterpret_cast<const char*>(meta_head + cur_qt * 64);
            uint32_t off = (uint32_t)lane * 4u;
            if (MASKED && wave > 0) {
                src = reinterpret_cast<const char*>((wave == 1 ? p.kv_start : p.kv_end) + (int64_t)b * p.Lq + r0);
                off = (uint32_t)min(l32, p.row_end - 1 - r0) * 4u;
            }
            dma4<RESTORED>(src, off, meta0 + (uint32_t)buf * META_B + (uint32_t)wave * 256u);
        }
        const uint32_t row0 = (uint32_t)min(r0 + ld_r, p.row_end - 1);
        const uint32_t row1 = (uint32_t)min(r0 + ld_r + 4, p.row_end - 1);
        const uint32_t slot = lds0 + (uint32_t)buf * (TILE_ELEMS * 2) + (uint32_t)slice * 2048u;
        dma16<RESTORED>(q_head, row0 * qrow_b + ld_c0, slot);
        dma16(q_head, row1 * qrow_b + ld_c1, slot + 1024);
        dma16<RESTORED>(do_head, row0 * dorow_b + ld_c0, slot + OFF_DO * 2);
        dma16(do_head, row1 * dorow_b + ld_c1, slot + OFF_DO * 2 + 1024);
    };
    auto advance = [&]() {   // next (head, row tile) of the walk, wrapping
        ++cur_qt;
        if (--cur_left > 0) return;
        if (++cur_run == 4 || sel4(cur_run, run_n) == 0) {
            cur_run = 0;
            if (++cur_gi == p.G) cur_gi = 0;
            enter_head();
        }
        cur_qt = sel4(cur_run, run_s);
        cur_left = sel4(cur_run, run_n);
    };

    // the finished dS^T tile goes to HBM as one contiguous 8 KB block
    auto copy_out = [&](const uint16_t* dst, int64_t ws_off) {
        const uint16_t *const r0 = dst + cp_rd[0] / 2, *const r1 = dst + cp_rd[1] / 2;
        const u32x2 a0 = lds_read_tr16(r0), a1 = lds_read_tr16(r1), c0 = lds_read_tr16(r0 + CP2 * BM), c1 = lds_read_tr16(r1 + CP2 * BM);
        const u32x4 a = {a0[0], a0[1], a1[0], a1[1]}, c2 = {c0[0], c0[1], c1[0], c1[1]};
        u32x4* const o = reinterpret_cast<u32x4*>(ws_lane + ws_off);
        if (p.ds_stream) {
            __builtin_nontemporal_store(a, o);
            __builtin_nontemporal_store(c2, o + CP2 * 4);
        } else {
            o[0] = a;
            o[CP2 * 4] = c2;
        }
    };

    // The work on a tile is spread over three steps so that, inside every wave, the
    // MFMAs of one tile and the VALU work of an earlier tile are independent and
    // overlap (on top of the overlap between the two waves of a SIMD):
    //   step i, P-wave: S(i) = Q K_w^T                     || P(i-1) = exp2(S(i-1)*c - LSE*log2e), masked
    //                   then hand P(i-1) over, dV_w^T += dO(i-1)^T P(i-1)
    //   step i, D-wave: dP(i-1) = dO V_w^T                 || dS(i-2) = P(i-2) (dP(i-2)*scale - delta*scale)
    //                   then dS^T(i-2) to LDS, dK_w^T += Q(i-2)^T dS(i-2)
    //   step i, all   : request tile i+2, copy dS^T(i-3) out
    // Flags say which halves exist at the edges of the walk; they are compile-time
    // constants in the steady-state loop.
    auto p_step = [&](auto tail_c, bool s_live, bool pv_live, const uint16_t* tile_cur, const uint16_t* tile_prev,
                      const u32x4* meta, uint16_t* pbuf, f32x16& s_carry, f32x16& bv, int64_t bias_off, int bias_r0)
                      __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail_c)::value;
        const char* qt = reinterpret_cast<const char*>(tile_cur);     // Q of tile i
        const char* dot = reinterpret_cast<const char*>(tile_prev);   // dO of tile i-1
        bf16x8 qa[8];
        u32x2 da[4][2][2];
        // MASKED: lane l looks at the key interval of row l of the previous tile (requested
        // first, so the answer is there long before it is needed)
        int iv_s = 0, iv_e = 0;
        if (MASKED && pv_live) {
            const int32_t* iv = reinterpret_cast<const int32_t*>(meta + 16);
            iv_s = iv[l32];
            iv_e = iv[64 + l32];
        }
        if (s_live) {
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk)
                qa[kk] = *reinterpret_cast<const bf16x8*>(qt + row_rd + ((uint32_t)(kk * 32) ^ row_h));
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x16 s_new;
        if (s_live) {
#pragma unroll
            for (int v = 0; v < 16; ++v) s_new[v] = 0.f;
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) s_new = E::mfma(qa[kk], breg[kk], s_new);
        }
        if (pv_live) {
            // dO^T operands: requested once the S operands are consumed; they land while
            // the exp2 phase runs in the shadow of the S MFMAs
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    da[dt][j][0] = lds_read_tr16(reinterpret_cast<const uint16_t*>(dot + t_rd[dt][0] + j * 4096));
                    da[dt][j][1] = lds_read_tr16(reinterpret_cast<const uint16_t*>(dot + t_rd[dt][1] + j * 4096));
                }
            f32x16 s = s_carry;
#pragma unroll
            for (int vg = 0; vg < 4; ++vg) {
                const f32x4 l4 = __builtin_bit_cast(f32x4, meta[2 * vg + g]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float off = BIAS ? fmaf(bv[4 * vg + r], LOG2E, -l4[r]) : -l4[r];
                    s[4 * vg + r] = __builtin_amdgcn_exp2f(fmaf(s[4 * vg + r], c, off));
                }
            }
            if (BIAS) __builtin_amdgcn_sched_barrier(0);
            if (MASKED) {
                // most (tile, token slice) pairs a mask leaves alive are alive as a whole; only a
                // slice that some row of the tile cuts is masked element by element
                const bool cut = iv_s > slice_lo || iv_e < slice_lo + 32;
                if (!slice_valid || __builtin_amdgcn_ballot_w64(cut) != 0) {
#pragma unroll
                    for (int vg = 0; vg < 4; ++vg) {
                        const u32x4 sp = meta[16 + 2 * vg + g];
                        const u32x4 ep = meta[32 + 2 * vg + g];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const bool vis = kv_valid && my_kv >= (int)sp[r] && my_kv < (int)ep[r];
                            s[4 * vg + r] = vis ? s[4 * vg + r] : 0.f;
                        }
                    }
                }
            } else if (TAIL) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = kv_valid ? s[v] : 0.f;
            }
            u32x4 pu[2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) pu[j][e] = E::pack(s[8 * j + 2 * e], s[8 * j + 2 * e + 1]);
            *reinterpret_cast<u32x4*>(pbuf + pb_off) = pu[0];
            *reinterpret_cast<u32x4*>(pbuf + pb_off + 64 * 8) = pu[1];
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const u32x4 a = {da[dt][j][0][0], da[dt][j][0][1], da[dt][j][1][0], da[dt][j][1][1]};
                    acc[dt] = E::mfma(as_bf16x8(a), as_bf16x8(pu[j]), acc[dt]);
                }
        }
        if (BIAS && s_live) {   // for the next step: bias of (row 8 vg + 4 g + r of this tile, the lane's token)
            const float* bp = p.bias + bias_off + min(my_kv, p.Lkv - 1);
            const int last = p.row_end - 1 - bias_r0;
#pragma unroll
            for (int v = 0; v < 16; ++v) bv[v] = bp[(int64_t)min(8 * (v >> 2) + 4 * g + (v & 3), last) * p.bias_r];
        }
        if (s_live) s_carry = s_new;
    };

    auto d_step = [&](bool pv_live, bool ds_live, const uint16_t* tile_p1, const uint16_t* tile_p2, const u32x4* meta,
                      const uint16_t* pbuf, uint16_t* dst, f32x16& dp_carry) __attribute__((always_inline)) {
        const char* dor = reinterpret_cast<const char*>(tile_p1);                    // dO rows of tile i-1
        const char* qt = reinterpret_cast<const char*>(tile_p2);                     // Q of tile i-2
        u32x4 pu[2];
        u32x2 qa[4][2][2];
        bf16x8 da[8];
        if (pv_live) {
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk)
                da[kk] = *reinterpret_cast<const bf16x8*>(dor + row_rd + ((uint32_t)(kk * 32) ^ row_h));
        }
        if (ds_live) {
            pu[0] = *reinterpret_cast<const u32x4*>(pbuf + pb_off);
            pu[1] = *reinterpret_cast<const u32x4*>(pbuf + pb_off + 64 * 8);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x16 dp_new;
        if (pv_live) {
#pragma unroll
            for (int v = 0; v < 16; ++v) dp_new[v] = 0.f;
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) dp_new = E::mfma(da[kk], breg[kk], dp_new);
        }
        if (ds_live) {
            // Q^T operands: requested once the dO operands are consumed
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    qa[dt][j][0] = lds_read_tr16(reinterpret_cast<const uint16_t*>(qt + t_rd[dt][0] + j * 4096));
                    qa[dt][j][1] = lds_read_tr16(reinterpret_cast<const uint16_t*>(qt + t_rd[dt][1] + j * 4096));
                }
            u32x4 dsu[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const f32x4 da4 = __builtin_bit_cast(f32x4, meta[8 + 4 * j + g]);       // rows 16j + 4g + 0..3
                const f32x4 db4 = __builtin_bit_cast(f32x4, meta[8 + 4 * j + 2 + g]);   // rows 16j + 8 + 4g + 0..3
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // registers 8j + 2e, 8j + 2e + 1 are rows 16j + 8(e/2) + 4g + 2(e%2) + {0, 1}
                    const float d0 = (e < 2) ? da4[2 * (e & 1)] : db4[2 * (e & 1)];
                    const float d1 = (e < 2) ? da4[2 * (e & 1) + 1] : db4[2 * (e & 1) + 1];
                    // scale * P * (dP - delta), with delta * scale from the record
                    dsu[j][e] = E::pack(E::lo(pu[j][e]) * fmaf(dp_carry[8 * j + 2 * e], p.scale, -d0),
                                          E::hi(pu[j][e]) * fmaf(dp_carry[8 * j + 2 * e + 1], p.scale, -d1));
                }
            }
            uint16_t* const dsp = dst + (32 * slice + l32) * BM + 4 * g;
#pragma unroll
            for (int vg = 0; vg < 4; ++vg) {
                const u32x2 w = {dsu[vg >> 1][2 * (vg & 1)], dsu[vg >> 1][2 * (vg & 1) + 1]};
                *reinterpret_cast<u32x2*>(dsp + 8 * (vg ^ ((l32 >> 2) & 3))) = w;
            }
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const u32x4 a = {qa[dt][j][0][0], qa[dt][j][0][1], qa[dt][j][1][0], qa[dt][j][1][1]};
                    acc[dt] = E::mfma(as_bf16x8(a), as_bf16x8(dsu[j]), acc[dt]);
                }
        }
        if (pv_live) dp_carry = dp_new;
    };

    // The loop exists once per role (no branch on the role inside it).
    auto run = [&](auto tail_c, auto role_c) {
        constexpr bool DROLE = decltype(role_c)::value;
        if (n_iter == 0) return;
        // tile i lives in qt(i % 6) / dot(i % 6) with its row metadata in meta_s4[i % 6]; P(i) in pbf(i & 1); dS^T(i) in dst(i & 1)
        auto qt = [&](int k) { return smem + OFF_Q + k * TILE_ELEMS; };
        auto dot = [&](int k) { return smem + OFF_DO + k * TILE_ELEMS; };
        auto dst = [&](int k) { return smem + OFF_DST + k * DST_ELEMS; };
        auto pbf = [&](int k) { return smem + OFF_PB + k * PB_ELEMS; };
        auto m6 = [](int x) { return x >= NQD ? x - NQD : x; };
        // dS^T workspace offsets of the tiles in flight: a tile enters at [5] when requested
        // (two steps ahead); at step i (before that step's shift) tile i is at [3], tile i-3 at [0]
        int64_t w_q[6] = {0, 0, 0, 0, 0, 0};
        int64_t b_q[6] = {0, 0, 0, 0, 0, 0};    // BIAS: offset of (b, h, first row of the tile) in the bias
        int r_q[6] = {0, 0, 0, 0, 0, 0};        // BIAS: first row of the tile
        auto fetch = [&](int buf) {   // start the loads of the next tile of the walk
            w_q[5] = ws_head + (int64_t)cur_qt * (BN * BM);
            if (BIAS) {
                r_q[5] = p.row_begin + cur_qt * BM;
                b_q[5] = b * p.bias_b + (hk * p.G + cur_gi) * p.bias_h + (int64_t)r_q[5] * p.bias_r;
            }
            if (!DROLE) prefetch(buf);
            advance();
        };
        auto shift = [&]() {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                w_q[k] = w_q[k + 1];
                if (BIAS) { b_q[k] = b_q[k + 1]; r_q[k] = r_q[k + 1]; }
            }
        };
        f32x16 carry;     // P-wave: raw S of the previous tile; D-wave: dP of the previous tile
#pragma unroll
        for (int v = 0; v < 16; ++v) carry[v] = 0.f;
        f32x16 bv = carry;      // BIAS, P-wave: of the previous tile, on its way since the step before
        int rc = 0;       // i % 6

        auto step = [&](int i, bool s_live, bool pv_live, bool ds_live, bool copy) __attribute__((always_inline)) {
            // A P-wave's part of tile i (requested two steps ago) must have landed.  Vector-memory
            // operations complete in issue order, and after the loads of tile i the wave has issued
            // at least: the 4 loads of tile i+1 (requested in step i-1, or in the prologue), and
            // from step 5 on also the 2 dS^T stores of step i-2 and the 2 of step i-1 (steps 0-2
            // store nothing; wave 0's metadata loads and the bias loads only add to this).  So "at
            // most 8 outstanding" (4 in the first steps) says tile i is there and leaves everything
            // younger in flight.
            if (!DROLE) {
                if (i + 1 >= n_iter) wait_vmcnt<0>();
                else if (i >= 5) wait_vmcnt<8>();
                else wait_vmcnt<4>();
            }
            lds_barrier();
            // the bias has come before the next tile is requested, or its wait would be for that as well
            if (BIAS && !DROLE) asm volatile("" : "+v"(bv));
            // tile i+2 replaces tile i-4, whose last readers finished long before this barrier
            if (i + 2 < n_iter) fetch(m6(rc + 2));
            const int r1 = m6(rc + 5), r2 = m6(rc + 4);     // (i - 1) % 6, (i - 2) % 6
            if (!DROLE)
                p_step(tail_c, s_live, pv_live, qt(rc), dot(r1), meta_s4[r1], pbf((i + 1) & 1), carry, bv, b_q[3], r_q[3]);
            else
                d_step(pv_live, ds_live, dot(r1), qt(r2), meta_s4[r2], pbf(i & 1), dst(i & 1), carry);
            // dS^T(i-3) to HBM last: its LDS read queues behind this step's operand reads
            // instead of delaying them, and only has to finish before the next barrier
            if (!DROLE && copy) copy_out(dst((i + 1) & 1), w_q[0]);
            shift();
            rc = m6(rc + 1);
        };
        fetch(0);
        shift();
        if (n_iter > 1) fetch(1);
        shift();
        const int last = n_iter + 1;
        int i = 0;
        for (; i < 3 && i <= last; ++i) step(i, i < n_iter, i >= 1 && i <= n_iter, i >= 2, false);
        // Steady state: steps 3 .. 3 + 6 trips - 1 (every one of them with all its parts alive and a tile to
        // request) run in the hand-scheduled loops of gen_bwd_loop.py, six steps a trip; the steps after
        // them continue below as if they had run here.  Left to the code above: heads of 32 and 16, a dense
        // bias without intervals per row (the host always has some: what the bias leaves visible), the last token block
        // where there is no mask, and token blocks whose live tiles are not one run.
        // The code above leaves the matrix pipe to the compiler's order and, masked, keeps its walk in spilled
        // scalar registers.  Forward and backward of an attention, us, that code against the loops: 2 x 3000 rows,
        // images of 3202 tokens 1423 -> 1199; 2 x 1023 rows x 6404 tokens 2039 -> 1999 (whole layer);
        // heads of 64, 2048 x 6404 708 -> 697.  With a dense bias (fp16, 16 heads, 1024 x 4096; bwd_kernel) 120 -> 109, and 106
        // since the steps left above have their bias on its way a step ahead of its use, too.
        if constexpr ((DH == 128 || DH == 64) && (MASKED || !BIAS) && !decltype(tail_c)::value) {
            int trips = uniform32((n_iter - 5) / 6);
            // a row of the bias in bytes is a factor of 24 bits there
            if (i == 3 && trips >= 1 && run_n[1] == 0 && (!BIAS || p.bias_r < (1 << 22))) {
                const int steps = 6 * trips;
                uint32_t ra[8], ta[8];      // with heads of 64 half of each stays unused
#pragma unroll
                for (int kk = 0; kk < 8; ++kk)
                    ra[kk] = lds0 + (DROLE ? OFF_DO : OFF_Q) * 2 + row_rd + ((uint32_t)(kk * 32) ^ row_h);
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) {
                    ta[2 * dt] = lds0 + (DROLE ? OFF_Q : OFF_DO) * 2 + t_rd[dt][0];
                    ta[2 * dt + 1] = lds0 + (DROLE ? OFF_Q : OFF_DO) * 2 + t_rd[dt][1];
                }
                const uint32_t a_pb = lds0 + OFF_PB * 2 + (uint32_t)pb_off * 2;
                const uint32_t a_meta = meta0 + (uint32_t)g * 16u;
                if constexpr (!DROLE) {
                    const uint32_t meta_w = wave < META_WAVES ? (uint32_t)wave * 256u : 0u;
                    uint16_t* ws_k = p.ds_ws + (int64_t)kblk * p.ws_ld;
                    const char* qp = uniform_ptr(q_head + (int64_t)(p.row_begin + cur_qt * BM) * qrow_b);
                    const char* dop = uniform_ptr(do_head + (int64_t)(p.row_begin + cur_qt * BM) * dorow_b);
                    const char* m_src = reinterpret_cast<const char*>(meta_head + cur_qt * 64);
                    if (meta_w) m_src = reinterpret_cast<const char*>((wave == 1 ? p.kv_start : p.kv_end) + (int64_t)b * p.Lq +
                                                                      p.row_begin + cur_qt * BM);
                    const char* mp = uniform_ptr(m_src);
                    const char* wn = uniform_ptr(reinterpret_cast<const char*>(ws_k + ws_head + (int64_t)cur_qt * (BN * BM)));
                    const char* w0 = uniform_ptr(reinterpret_cast<const char*>(ws_k + w_q[0]));
                    const char* w1 = uniform_ptr(reinterpret_cast<const char*>(ws_k + w_q[1]));
                    const char* w2 = uniform_ptr(reinterpret_cast<const char*>(ws_k + w_q[2]));
                    const char* w3 = uniform_ptr(reinterpret_cast<const char*>(ws_k + w_q[3]));
                    const char* w4 = uniform_ptr(reinterpret_cast<const char*>(ws_k + w_q[4]));
                    const char* w5 = w4;
                    int left = uniform32(cur_left);
                    const int64_t hdq = uniform64((int64_t)p.qs.h * 2 - (int64_t)n_live * BM * qrow_b);
                    const int64_t hddo = uniform64((int64_t)p.dos.h * 2 - (int64_t)n_live * BM * dorow_b);
                    const int64_t hdws = uniform64((int64_t)p.ws_bh * 2 - (int64_t)n_live * (BN * BM * 2));
                    const int64_t hdm = uniform64(meta_w ? -(int64_t)n_live * (BM * 4) : (int64_t)(n_qtiles - n_live) * 256);
                    const uint32_t a_cp0 = lds0 + OFF_DST * 2 + cp_rd[0], a_cp1 = lds0 + OFF_DST * 2 + cp_rd[1];
                    const uint32_t g_cp = (uint32_t)(128 * slice + lane) * 16;
                    // the four loads of a tile; in a window's last one the rows end at `last`
                    const int last = (p.row_end - p.row_begin - 1) % BM;
                    const bool ragged = last != BM - 1 && run_s[0] + n_live == n_qtiles;
                    const int lr = (lane >> 4) + 8 * slice;
                    const uint32_t past0 = (uint32_t)max(lr - last, 0), past1 = (uint32_t)max(lr + 4 - last, 0);
                    const bool now = ragged && left == 1;       // the first tile to request is such a tile
                    const uint32_t rl0 = (uint32_t)lr - (now ? past0 : 0u), rl1 = (uint32_t)(lr + 4) - (now ? past1 : 0u);
                    uint32_t g_t[4] = {rl0 * qrow_b + ld_c0, rl1 * qrow_b + ld_c1, rl0 * dorow_b + ld_c0, rl1 * dorow_b + ld_c1};
                    const uint32_t past_iv = meta_w ? (uint32_t)max(l32 - last, 0) * 4u : 0u;
                    uint32_t g_meta = (meta_w ? (uint32_t)l32 : (uint32_t)lane) * 4u - (now ? past_iv : 0u);
                    const uint32_t a_iv = meta0 + 256u + (uint32_t)l32 * 4u;
                    const int token = kv_valid ? my_kv : 0x7fffffff;
                    // bias: of tile i - 1 in registers, of tile i on its way to LDS, of tile i + 1 the first the loop requests
                    const uint32_t brow_b = (uint32_t)p.bias_r * 4u;
                    const uint32_t lds_bias = lds0 + OFF_BIAS * 2 + (uint32_t)slice * 4096u;
                    const uint32_t b_row = 4u * ((lane >> 3) & 1) + (lane >> 4);
                    // 16 bytes of a row, the last of the row for lanes past it
                    const uint32_t b_chunk = (uint32_t)min(slice_lo + 4 * (lane & 7), (p.Lkv - 1) & ~3) * 4u;
                    const uint32_t a_bias = lds_bias + (uint32_t)g * 128u + (uint32_t)l32 * 4u;
                    const char* bp = nullptr;
                    int b_left = 0;
                    int64_t hdb = 0;
                    if constexpr (BIAS) {
                        const char* b0 = uniform_ptr(reinterpret_cast<const char*>(p.bias + b_q[3]));
#pragma unroll
                        for (int n = 0; n < 4; ++n)
                            dma16<RESTORED>(b0, (uint32_t)min((int)b_row + 8 * n, p.row_end - 1 - r_q[3]) * brow_b + b_chunk,
                                            lds_bias + 1024u * n);
                        bp = uniform_ptr(reinterpret_cast<const char*>(p.bias + b_q[4]));
                        b_left = uniform32(n_live - (it_lo + i + 1) % n_live);
                        hdb = uniform64((int64_t)p.bias_h * 4 - (int64_t)n_live * BM * brow_b);
                    }
                    wait_vmcnt<4>();    // tile 3 (the loads of tile 4 may be in flight); the loop counts from there
                    if constexpr (BIAS && !F16 && DH == 128) {
                        asm volatile(
#include "lvx_bwd_loop_p_bf16_128_bias.inc"
                            LVX_BWD_P_BIAS_OPERANDS);
                    } else if constexpr (BIAS && !F16) {
                        asm volatile(
#include "lvx_bwd_loop_p_bf16_64_bias.inc"
                            LVX_BWD_P_BIAS_OPERANDS);
                    } else if constexpr (BIAS && DH == 128) {
                        asm volatile(
#include "lvx_bwd_loop_p_f16_128_bias.inc"
                            LVX_BWD_P_BIAS_OPERANDS);
                    } else if constexpr (BIAS) {
                        asm volatile(
#include "lvx_bwd_loop_p_f16_64_bias.inc"
                            LVX_BWD_P_BIAS_OPERANDS);
                    } else if constexpr (!F16 && DH == 128 && !MASKED) {
                        asm volatile(
#include "lvx_bwd_loop_p_bf16_128_plain.inc"
                            LVX_BWD_P_OPERANDS);
                    } else if constexpr (!F16 && DH == 128) {
                        asm volatile(
#include "lvx_bwd_loop_p_bf16_128_masked.inc"
                            LVX_BWD_P_OPERANDS);
                    } else if constexpr (!F16 && !MASKED) {
                        asm volatile(
#include "lvx_bwd_loop_p_bf16_64_plain.inc"
                            LVX_BWD_P_OPERANDS);
                    } else if constexpr (!F16) {
                        asm volatile(
#include "lvx_bwd_loop_p_bf16_64_masked.inc"
                            LVX_BWD_P_OPERANDS);
                    } else if constexpr (DH == 128 && !MASKED) {
                        asm volatile(
#include "lvx_bwd_loop_p_f16_128_plain.inc"
                            LVX_BWD_P_OPERANDS);
                    } else if constexpr (DH == 128) {
                        asm volatile(
#include "lvx_bwd_loop_p_f16_128_masked.inc"
                            LVX_BWD_P_OPERANDS);
                    } else if constexpr (!MASKED) {
                        asm volatile(
#include "lvx_bwd_loop_p_f16_64_plain.inc"
                            LVX_BWD_P_OPERANDS);
                    } else {
                        asm volatile(
#include "lvx_bwd_loop_p_f16_64_masked.inc"
                            LVX_BWD_P_OPERANDS);
                    }
                    wait_vmcnt<0>();    // the steps below count the operations in flight from scratch
                    w_q[0] = reinterpret_cast<const uint16_t*>(w0) - ws_k;
                    w_q[1] = reinterpret_cast<const uint16_t*>(w1) - ws_k;
                    w_q[2] = reinterpret_cast<const uint16_t*>(w2) - ws_k;
                    w_q[3] = reinterpret_cast<const uint16_t*>(w3) - ws_k;
                    w_q[4] = reinterpret_cast<const uint16_t*>(w4) - ws_k;
                } else {
                    uint32_t a_ds[4];
#pragma unroll
                    for (int vg = 0; vg < 4; ++vg)
                        a_ds[vg] = lds0 + OFF_DST * 2 + (uint32_t)((32 * slice + l32) * BM + 8 * (vg ^ ((l32 >> 2) & 3)) + 4 * g) * 2;
                    if constexpr (!F16 && DH == 128) {
                        asm volatile(
#include "lvx_bwd_loop_d_bf16_128.inc"
                            LVX_BWD_D_OPERANDS);
                    } else if constexpr (!F16) {
                        asm volatile(
#include "lvx_bwd_loop_d_bf16_64.inc"
                            LVX_BWD_D_OPERANDS);
                    } else if constexpr (DH == 128) {
                        asm volatile(
#include "lvx_bwd_loop_d_f16_128.inc"
                            LVX_BWD_D_OPERANDS);
                    } else {
                        asm volatile(
#include "lvx_bwd_loop_d_f16_64.inc"
                            LVX_BWD_D_OPERANDS);
                    }
                }
                i += steps;
                if (BIAS) {     // tiles i-1 .. i+1
#pragma unroll
                    for (int k = 2; k < 5; ++k) {
                        const int pos = it_lo + i - 3 + k;
                        r_q[k] = p.row_begin + (run_s[0] + pos % n_live) * BM;
                        b_q[k] = b * p.bias_b + (hk * p.G + pos / n_live) * p.bias_h + (int64_t)r_q[k] * p.bias_r;
                    }
                }
                // the walk stands at the tile after the last one requested
                const int pos = it_lo + i + 2;
                cur_gi = pos / n_live;
                cur_run = 0;
                cur_qt = run_s[0] + pos % n_live;
                cur_left = n_live - pos % n_live;
                if (cur_gi >= p.G) cur_gi = 0;
                enter_head();
            }
        }
        for (; i < n_iter; ++i) step(i, true, true, true, true);
        for (; i <= last; ++i) step(i, false, i <= n_iter, true, true);
        __syncthreads();
        if (!DROLE) copy_out(dst((n_iter - 1) & 1), w_q[0]);
    };
    if (d_role) {
        if (!MASKED && tail_block) run(std::true_type{}, std::true_type{});
        else run(std::false_type{}, std::true_type{});
    } else {
        if (!MASKED && tail_block) run(std::true_type{}, std::false_type{});
        else run(std::false_type{}, std::false_type{});
    }

    // ---- epilogue: rows of acc = head-dim, cols = this wave's tokens; P-waves hold dV^T, D-waves dK^T.
    // A lane holds 4 consecutive values of d of one token per register group.  The accumulator is turned through LDS, in
    // the type it leaves in, so that the lanes of an instruction cover whole token rows; rows are 16 bytes longer there
    // than their values, as in the forward.  Stored from the registers, 16 or 32 bytes of 32 rows at a time, adding to an
    // fp32 accumulator took 9.5 us at the end of a work-group of 32 steps (46 us in all) and 16-bit rows 3 - 5; so 7.5 -
    // all CUs at once then move 67 MB, 9 TB/s; lines brought into the L2 ahead of it cost the steps what they save
    // here - and 1.2 - 1.7.
    __syncthreads();   // the staging buffers are free now
    constexpr int EP32 = 4 * DH + 16, EP16 = 2 * DH + 16;
    static_assert(8 * 32 * EP32 <= SMEM_ELEMS * 2);
    char* const ep = reinterpret_cast<char*>(smem) + wave * (32 * EP32);
    const int n_tok = p.Lkv - slice_lo;                 // of this wave's 32 tokens those that exist, where fewer
    if (n_tok <= 0) return;
    const Strides3 os = alone ? (d_role ? p.dks_whole : p.dvs_whole) : (d_role ? p.dks : p.dvs);
    void* const optr = alone ? (d_role ? p.dk_whole : p.dv_whole) : (d_role ? p.dk : p.dv);
    const int64_t o_at = b * os.b + hk * os.h + (int64_t)slice_lo * os.s;
    auto turn_f32 = [&]() {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int vg = 0; vg < 4; ++vg) {
                if (dt * 32 + 8 * vg >= DH) continue;   // only with DH = 16
                const f32x4 x = {acc[dt][4 * vg], acc[dt][4 * vg + 1], acc[dt][4 * vg + 2], acc[dt][4 * vg + 3]};
                *reinterpret_cast<f32x4*>(ep + l32 * EP32 + g * 16 + (8 * dt + 2 * vg) * 16) = x;
            }
        wait_lds();     // this wave's rows are its own
    };
    if (dkv_mode == 2) {
        // Several work-groups (ranges of steps) share this token block: atomic adds, 64 consecutive floats
        // (two full lines) of one token row each
        if (n_iter == 0) return;
        turn_f32();
        float* const op = reinterpret_cast<float*>(optr) + o_at + lane;
        const float* const src = reinterpret_cast<const float*>(ep) + lane;
        for (int t = 0; t < min(n_tok, 32); ++t) {
            if (DH >= 64 || lane < DH) unsafeAtomicAdd(op + t * os.s, src[t * (EP32 / 4)]);
            if (DH == 128) unsafeAtomicAdd(op + t * os.s + 64, src[t * (EP32 / 4) + 64]);
        }
    } else if (dkv_mode == 3) {
        // A range of a block that has several: its slice, whole lines per instruction
        constexpr int CPF = DH / 4, RPS = 64 / CPF;
        turn_f32();
        uint32_t id = blockIdx.x;           // taken apart once more: no scalar is to live through the steps for it
        asm volatile("" : "+s"(id));
        const int x = (int)(id % 8), at = x * p.per_xcd + (int)(id / 8);
        int64_t range_slice = at - min(p.whole_blocks, p.n_blocks - x * p.blocks_per_xcd);
        if (MASKED && p.plan) {
            const uint32_t* const e = p.plan + (int64_t)at * PLAN_ENTRY;
            range_slice = e[1] + (e[0] >> 24);
        }
        float* const op = p.slices + range_slice * (2 * BN * DH) + (d_role ? 0 : BN * DH) + (32 * slice + lane / CPF) * DH + (lane % CPF) * 4;
#pragma unroll
        for (int i = 0; i < 32 / RPS; ++i)
            *reinterpret_cast<f32x4*>(op + i * RPS * DH) = *reinterpret_cast<const f32x4*>(ep + (lane / CPF) * EP32 + (lane % CPF) * 16 + i * (RPS * EP32));
    } else if (dkv_mode == 1) {
        constexpr int CPF = DH / 4, RPS = 64 / CPF;     // chunks of a row of floats, rows per instruction
        float* const op = reinterpret_cast<float*>(optr) + o_at + (lane % CPF) * 4;
        f32x4 old[32 / RPS];                            // on their way while the accumulator is turned
#pragma unroll
        for (int i = 0; i < 32 / RPS; ++i) old[i] = *reinterpret_cast<const f32x4*>(op + min(i * RPS + lane / CPF, n_tok - 1) * os.s);
        turn_f32();
#pragma unroll
        for (int i = 0; i < 32 / RPS; ++i) {
            const int t = i * RPS + lane / CPF;
            const f32x4 x = *reinterpret_cast<const f32x4*>(ep + (lane / CPF) * EP32 + (lane % CPF) * 16 + i * (RPS * EP32));
            if (t < n_tok) *reinterpret_cast<f32x4*>(op + t * os.s) = old[i] + x;
        }
    } else {
        constexpr int CPR = DH / 8, RPS = 64 / CPR;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int vg = 0; vg < 4; ++vg) {
                if (dt * 32 + 8 * vg >= DH) continue;   // only with DH = 16
                u32x2 a;
                a[0] = E::pack(acc[dt][4 * vg], acc[dt][4 * vg + 1]);
                a[1] = E::pack(acc[dt][4 * vg + 2], acc[dt][4 * vg + 3]);
                // of rows 16 apart one has the halves of its chunks exchanged: conflict-free
                *reinterpret_cast<u32x2*>(ep + l32 * EP16 + ((g ^ (l32 >> 4)) << 3) + (4 * dt + vg) * 16) = a;
            }
        wait_lds();
        uint16_t* const op = reinterpret_cast<uint16_t*>(optr) + o_at + (lane % CPR) * 8;
#pragma unroll
        for (int i = 0; i < 32 / RPS; ++i) {
            const int t = i * RPS + lane / CPR;
            const u32x4 x = *reinterpret_cast<const u32x4*>(ep + (lane / CPR) * EP16 + (lane % CPR) * 16 + i * (RPS * EP16));
            const u32x4 y = (t >> 4) & 1 ? u32x4{x[2], x[3], x[0], x[1]} : x;
            if (t < n_tok) *reinterpret_cast<u32x4*>(op + t * os.s) = y;
        }
    }
}

}  // namespace

namespace {
template <int DH, bool F16>
hipError_t launch_bwd_t(const BwdParams& p, bool masked, hipStream_t st) {
    const int grid = p.own_wg + 8 * p.dq_before.blocks_per_xcd;
    if (p.bias) {
        if (masked) return launch1((bwd_kernel<DH, true, true, F16>), dim3(grid), dim3(NT), st, p);
        else return launch1((bwd_kernel<DH, false, true, F16>), dim3(grid), dim3(NT), st, p);
    } else {
        if (masked) return launch1((bwd_kernel<DH, true, false, F16>), dim3(grid), dim3(NT), st, p);
        else return launch1((bwd_kernel<DH, false, false, F16>), dim3(grid), dim3(NT), st, p);
    }
}
}  // namespace

hipError_t launch_bwd(const BwdParams& params, bool masked, hipStream_t st, const CastParams* dq_before) {
    BwdParams p = params;
    p.own_wg = p.plan ? 8 * p.per_xcd : 8 * (p.whole_blocks + p.mid_blocks * p.q_splits + (p.blocks_per_xcd - p.whole_blocks - p.mid_blocks) * p.q_splits2);
    p.dq_before = CastParams{};
    if (dq_before) {
        p.dq_before = *dq_before;
        const hipError_t e = plan_cast_t(p.dq_before, NT);
        if (e != hipSuccess) return e;
    }
    p.by_splits = divisor(p.q_splits);
    p.by_splits2 = divisor(p.q_splits2);
    p.by_kv_blocks = divisor(p.n_kv_blocks);
    p.by_B = divisor(p.B);
    switch (p.D) {
        case 16: return p.f16 ? launch_bwd_t<16, true>(p, masked, st) : launch_bwd_t<16, false>(p, masked, st);
        case 32: return p.f16 ? launch_bwd_t<32, true>(p, masked, st) : launch_bwd_t<32, false>(p, masked, st);
        case 64: return p.f16 ? launch_bwd_t<64, true>(p, masked, st) : launch_bwd_t<64, false>(p, masked, st);
        case 128: return p.f16 ? launch_bwd_t<128, true>(p, masked, st) : launch_bwd_t<128, false>(p, masked, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace lvx

// bf16 GEMM for the K/V recompute (K = X W_k, V = X W_v), its input gradient
// (dX = dK W_k^T + dV W_v^T, one GEMM whose contraction runs over two operand
// pairs) and the weight gradients (dW = X^T dK).  fp32 accumulate on v_mfma_f32_32x32x16_bf16, bf16 output.
//
// Structure (8 waves, two per SIMD, in lock-step "ping-pong"):
//  * Operand tiles go from global memory straight into LDS with
//    global_load_lds_dwordx4 (no staging registers), NS stages of 32 k deep, so
//    a tile is requested NS-1 stages before it is used.
//  * Waves 0-3 and waves 4-7 (one of each per SIMD) run the same loop half a
//    stage apart: while one set issues the 16 MFMAs of a stage from registers,
//    the other set fetches its operands of the next stage from LDS and issues
//    its share of the global loads; a work-group barrier after every phase
//    keeps the two sets alternating, so the MFMA pipe of every SIMD always has
//    one wave feeding it and the LDS / memory latency of the other is hidden.
//  * The direct-to-LDS load writes 64 lanes x 16 bytes contiguously, so tiles
//    cannot be padded; bank conflicts are avoided by permuting 16-byte chunks
//    (an XOR of the chunk index with row bits), applied on the global-address
//    side when loading and on the LDS-address side when reading.
//  * An operand whose memory has the contraction index contiguous is read
//    with 16-byte LDS reads; one whose memory has the OTHER index contiguous
//    is kept as it lies, [k][rows], and read with the transposing LDS read.
//  * The MFMA computes C^T (A operand = rows of the B tile), so a lane ends up
//    with 4 consecutive columns of one C row and stores 8 bytes.
#include <type_traits>

#include "lvx_common.hpp"
#include "lvx_gemm_tiles.hpp"
#include "lvx_kernels.hpp"

namespace lvx {

namespace {

constexpr int BK = 32;                 // contraction depth of one stage
__device__ uint32_t zero_chunk[4];     // source of the chunks past the end of a contraction

__device__ __forceinline__ void phase_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// One operand's part of a stage: ROWS rows x 32 k, unpadded, in wave-chunks of
// 1 KiB (what one global_load_lds_dwordx4 writes).
//   !ROW_CONTIG (memory [row][k]): LDS row r at r*64 B; its 16-byte chunk c
//       (k = 8c..8c+7) sits at position c ^ ((r >> 2) & 3).
//    ROW_CONTIG (memory [k][row]): LDS k-row at k*ROWS*2 B; its chunk q (rows
//       8q..8q+7) sits at position q ^ ((k & 3) << 2).
template <bool ROW_CONTIG, int ROWS>
struct Region {
    static constexpr int BYTES = ROWS * BK * 2;
    static constexpr int CHUNKS = BYTES / 1024;
    static constexpr int LPR = ROWS / 8;          // lanes per k-row (ROW_CONTIG)

    // what lane `lane` of the wave loading chunk `ch` fetches: byte offset from the
    // stage base of the operand, and the k position inside the stage
    __device__ __forceinline__ static uint32_t src(int ch, int lane, int r0, int R, int64_t ld, int& kpos) {
        if (!ROW_CONTIG) {
            const int row = 16 * ch + (lane >> 2);
            const int c = (lane & 3) ^ ((lane >> 4) & 3);
            kpos = c * 8;
            return (uint32_t)(min(r0 + row, R - 1) - r0) * (uint32_t)ld * 2u + (uint32_t)c * 16u;
        }
        const int k = ch * (64 / LPR) + lane / LPR;
        const int q = (lane % LPR) ^ ((k & 3) << 2);
        kpos = k;
        const int r = min(r0 + q * 8, R - 8);
        return (uint32_t)k * (uint32_t)ld * 2u + (uint32_t)(r - r0) * 2u;
    }

    // per-lane LDS byte offsets for the operand reads of a wave whose first
    // 32-row tile in the region is tile j0 (W tiles per wave).
    //  !ROW_CONTIG: rd[kk] for k-step kk; add tile * 2048
    //   ROW_CONTIG: rd[t] for tile t; add kk * 16 * ROWS * 2 (+ 4 * ROWS * 2 for the second half)
    template <int W>
    __device__ __forceinline__ static void read_offsets(uint32_t* rd, int j0, int lane) {
        if (!ROW_CONTIG) {
            const int l32 = lane & 31, g = lane >> 5, s = (l32 >> 2) & 3;
            rd[0] = (uint32_t)(j0 * 2048 + l32 * 64 + ((g ^ s) * 16));
            rd[1] = (uint32_t)(j0 * 2048 + l32 * 64 + (((2 + g) ^ s) * 16));
        } else {
            const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1, g = lane >> 5;
#pragma unroll
            for (int i = 0; i < W; ++i)
                rd[i] = (uint32_t)((8 * g + r) * ROWS * 2 + 64 * ((j0 + i) ^ r) + (2 * u + (t >> 1)) * 16 + (t & 1) * 8);
        }
    }
    static constexpr int NRD(int W) { return ROW_CONTIG ? W : 2; }

    // operand (tile t of the wave, k-step kk) from the stage at LDS byte offset `base`
    __device__ __forceinline__ static bf16x8 operand(const char* lds, uint32_t base, const uint32_t* rd, int t, int kk) {
        if (!ROW_CONTIG) return *reinterpret_cast<const bf16x8*>(lds + base + rd[kk] + t * 2048);
        const uint16_t* p = reinterpret_cast<const uint16_t*>(lds + base + rd[t] + kk * 16 * ROWS * 2);
        return lds_operand_tr(p, 4 * ROWS);
    }
};

// GM x GN waves, each WM x WN MFMA tiles: work-group tile (32 WM GM) x (32 WN GN).
template <bool A_MCONTIG, bool B_NCONTIG, int GM, int GN, int WM, int WN, int NS, bool F16>
__global__ __launch_bounds__(512, 1) void gemm_kernel(const GemmParams p) {
    using E = Elt<F16>;
    static_assert(GM * GN == 8, "8 waves");
    constexpr int TM = 32 * WM * GM, TN = 32 * WN * GN;
    using RA = Region<A_MCONTIG, TM>;
    using RB = Region<B_NCONTIG, TN>;
    constexpr int STAGE = RA::BYTES + RB::BYTES;
    constexpr int LPG = (RA::CHUNKS + RB::CHUNKS) / 8;     // loads per wave per stage
    constexpr int LPG_A = RA::CHUNKS / 8;
    static_assert(RA::CHUNKS % 8 == 0 && RB::CHUNKS % 8 == 0, "chunks split evenly over 8 waves");
    constexpr int NRA = RA::NRD(WM), NRB = RB::NRD(WN);
    __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE];

    fetch_kernargs<sizeof(GemmParams)>();
    const int wid = xcd_remap(blockIdx.x, p.total_wg);
    if (wid >= p.total_wg) return;
    uint32_t tn, tm;
    const uint32_t prob = p.by_tiles_m.split(p.by_tiles_n.split(wid, tn), tm);
    const GemmProblem& pr = p.prob[prob];
    const int m0 = tm * TM, n0 = tn * TN;
    const int klen0 = pr.K[0];
    const int klen1 = pr.nseg > 1 ? pr.K[1] : 0;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int set = wave >> 2;
    const int wm = wave % GM, wn = wave / GM;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

    // ---- global -> LDS: this wave's LPG chunks of every stage
    const int64_t lda = pr.lda[0], ldb = pr.ldb[0];
    uint32_t voff[LPG];
    int kpos[LPG];
#pragma unroll
    for (int j = 0; j < LPG; ++j) {
        const int ch = wave + 8 * j;
        if (j < LPG_A) voff[j] = RA::src(ch, lane, m0, p.M, lda, kpos[j]);
        else voff[j] = RB::src(ch - RA::CHUNKS, lane, n0, p.N, ldb, kpos[j]);
    }
    const char* abase[2];
    const char* bbase[2];
#pragma unroll
    for (int sg = 0; sg < 2; ++sg) {
        const int ss = sg < pr.nseg ? sg : 0;
        abase[sg] = reinterpret_cast<const char*>(pr.A[ss]) + (A_MCONTIG ? (int64_t)m0 : (int64_t)m0 * lda) * 2;
        bbase[sg] = reinterpret_cast<const char*>(pr.Bm[ss]) + (B_NCONTIG ? (int64_t)n0 : (int64_t)n0 * ldb) * 2;
    }
    const int64_t a_kstride = A_MCONTIG ? lda * BK * 2 : BK * 2;   // bytes per stage
    const int64_t b_kstride = B_NCONTIG ? ldb * BK * 2 : BK * 2;
    const int steps0 = (klen0 + BK - 1) / BK;
    const int steps = steps0 + (klen1 + BK - 1) / BK;

    auto issue = [&](int s) {     // loads of stage s into ring slot s % NS
        const int sg = s >= steps0 ? 1 : 0;
        const int ks = sg ? s - steps0 : s;            // stage inside the operand
        const int krem = (sg ? klen1 : klen0) - ks * BK;
        const char* const ab = abase[sg] + ks * a_kstride;
        const char* const bb = bbase[sg] + ks * b_kstride;
        const uint32_t slot = lds0 + (uint32_t)(s % NS) * STAGE + (uint32_t)wave * 1024u;
        if (krem >= BK) {
#pragma unroll
            for (int j = 0; j < LPG; ++j)
                dma16(j < LPG_A ? ab : bb, voff[j], slot + (j < LPG_A ? j * 8192 : RA::BYTES + (j - LPG_A) * 8192));
        } else {
            const char* zc = reinterpret_cast<const char*>(zero_chunk);
#pragma unroll
            for (int j = 0; j < LPG; ++j) {
                const char* src = (j < LPG_A ? ab : bb) + voff[j];
                dma16_addr(kpos[j] < krem ? src : zc, slot + (j < LPG_A ? j * 8192 : RA::BYTES + (j - LPG_A) * 8192));
            }
        }
    };

    // ---- LDS -> registers
    uint32_t rda[NRA], rdb[NRB];
    RA::template read_offsets<WM>(rda, WM * wm, lane);
    RB::template read_offsets<WN>(rdb, WN * wn, lane);

    f32x16 acc[WN][WM];   // [n tile][m tile]
#pragma unroll
    for (int a = 0; a < WN; ++a)
#pragma unroll
        for (int b = 0; b < WM; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

    // prologue: stages 0 .. NS-2 in flight, stage 0 landed
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < steps) issue(s);
    if (steps > NS - 2) wait_vmcnt<(NS - 2) * LPG>();
    else wait_vmcnt<0>();
    phase_barrier();
    if (set == 1) phase_barrier();        // waves 4-7 run half a stage behind waves 0-3

    for (int s = 0; s < steps; ++s) {
        // memory phase: request stage s+NS-1, fetch this wave's operands of stage s
        if (s + NS - 1 < steps) issue(s + NS - 1);
        const uint32_t base = (uint32_t)(s % NS) * STAGE;
        bf16x8 am[2][WM], bn[2][WN];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
            for (int t = 0; t < WM; ++t) am[kk][t] = RA::operand(lds, base, rda, t, kk);
#pragma unroll
            for (int t = 0; t < WN; ++t) bn[kk][t] = RB::operand(lds, base + RA::BYTES, rdb, t, kk);
        }
        wait_lds();     // the slot may be overwritten once the next barrier is passed
        if (set == 1) {                     // stage s+1 must have landed before waves 0-3 read it
            if (s + NS - 1 < steps) wait_vmcnt<(NS - 2) * LPG>();
            else wait_vmcnt<0>();
        }
        phase_barrier();
        // compute phase
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int nt = 0; nt < WN; ++nt)
#pragma unroll
                for (int mt = 0; mt < WM; ++mt) acc[nt][mt] = E::mfma(bn[kk][nt], am[kk][mt], acc[nt][mt]);
        __builtin_amdgcn_s_setprio(0);
        if (set == 0) {
            if (s + NS - 1 < steps) wait_vmcnt<(NS - 2) * LPG>();
            else wait_vmcnt<0>();
        }
        phase_barrier();
    }
    if (set == 0) phase_barrier();

    // C^T tile: accumulator rows = n, cols = m
    // A lane holds 4 consecutive columns of one C row, so storing from the registers writes 8
    // bytes per lane into 32 different rows per instruction.  The rows go through the stage buffers
    // (free by now) instead, 256 at a time, and leave as whole row segments (TN * 2 bytes; N is a
    // multiple of 8), 16 bytes per lane.  16-byte chunk c of row r sits at position
    // c ^ (r mod chunks per row), with its two 8-byte halves exchanged in rows where bits 3 and 4 differ: the 32 rows a half-wave's 8-byte writes touch then land in different
    // chunks or, where they share a chunk position or banks (positions 8 or 16 apart), in
    // different halves; a read instruction takes whole rows.  Both are conflict-free.
    // `pair(mt, nt, vg)`: the 4 values of accumulator tile (nt, mt), register group vg, as two
    // packed words.
    constexpr int CPR = TN / 8;                 // 16-byte chunks per row
    static_assert((TN == 256 || TN == 128) && TM % 256 == 0 && 256 * TN * 2 <= NS * STAGE, "256 rows of the tile fit the stages");
    auto store_via_lds = [&](auto pair, uint16_t* dst) __attribute__((always_inline)) {
#pragma unroll
        for (int pass = 0; pass < TM / 256; ++pass) {
            __syncthreads();                    // every wave is done with what the buffers held
#pragma unroll
            for (int mt = 0; mt < WM; ++mt) {
                if (((WM * wm + mt) >> 3) != pass) continue;
#pragma unroll
                for (int nt = 0; nt < WN; ++nt)
#pragma unroll
                    for (int vg = 0; vg < 4; ++vg) {
                        const int ml = 32 * ((WM * wm + mt) & 7) + l32;
                        const int c = 4 * (WN * wn + nt) + vg;
                        *reinterpret_cast<u32x2*>(lds + ml * (TN * 2) + ((c ^ (l32 & (CPR - 1))) << 4) +
                                                  ((g ^ ((l32 >> 3) & 1) ^ (l32 >> 4)) << 3)) = pair(mt, nt, vg);
                    }
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < CPR / 2; ++i) {
                const int row = i * (512 / CPR) + tid / CPR, cc = tid % CPR;
                u32x4 val = *reinterpret_cast<const u32x4*>(lds + row * (TN * 2) + ((cc ^ (row & (CPR - 1))) << 4));
                if (((row >> 3) ^ (row >> 4)) & 1) val = u32x4{val[2], val[3], val[0], val[1]};
                const int m = m0 + 256 * pass + row, n = n0 + cc * 8;
                // (a streaming store: nobody on this CU reads the tile again)
                if (m < p.M && n < p.N) __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(dst + (int64_t)m * pr.ldc + n));
            }
        }
    };
    if (p.norm_w && prob == 0) {
        // RMS norm over each 128-column group (N and the tile are multiples of 128): the
        // group's columns sit in HW = 4 / WN waves with consecutive wn; row sums of squares
        // are exchanged through LDS, which no wave reads any more.
        constexpr int HW = 4 / WN;
        static_assert(WN == 2 || WN == 4, "a 128-column group spans 1 or 2 waves");
        float* const red = reinterpret_cast<float*>(lds);
        float rs[WM];
#pragma unroll
        for (int mt = 0; mt < WM; ++mt) {
            float ss = 0.f;
#pragma unroll
            for (int nt = 0; nt < WN; ++nt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float x = E::hi(E::pack(0.f, acc[nt][mt][i]));   // the product as bf16
                    acc[nt][mt][i] = x;
                    ss = fmaf(x, x, ss);
                }
            ss += __shfl_xor(ss, 32);
            rs[mt] = ss;
            if (HW > 1 && g == 0) red[(wave * WM + mt) * 32 + l32] = ss;
        }
        if (HW > 1) {
            __syncthreads();
            const int pw = wm + GM * (wn ^ 1);
#pragma unroll
            for (int mt = 0; mt < WM; ++mt) rs[mt] += red[(pw * WM + mt) * 32 + l32];
        }
        const int groups = p.N >> 7;
        // (N is a multiple of 128 here)
        float rr[WM];
#pragma unroll
        for (int mt = 0; mt < WM; ++mt) {
            const int m = m0 + 32 * (WM * wm + mt) + l32;
            rr[mt] = rsqrtf(rs[mt] * (1.f / 128.f) + p.norm_eps);
            const int ncol = n0 + 32 * WN * wn;
            if (m < p.M && p.rstd && g == 0 && (wn & (HW - 1)) == 0 && ncol < p.N) p.rstd[(int64_t)m * groups + (ncol >> 7)] = rr[mt];
        }
        if (p.c_raw)
            store_via_lds([&](int mt, int nt, int vg) {
                u32x2 w;
                w[0] = E::pack(acc[nt][mt][4 * vg], acc[nt][mt][4 * vg + 1]);
                w[1] = E::pack(acc[nt][mt][4 * vg + 2], acc[nt][mt][4 * vg + 3]);
                return w;
            }, p.c_raw);
        store_via_lds([&](int mt, int nt, int vg) {
            const int n = 32 * (WN * wn + nt) + 8 * vg + 4 * g;       // n0 is a multiple of 128
            const u32x2 wt = *reinterpret_cast<const u32x2*>(p.norm_w + (n & 127));
            const float r = rr[mt];
            const u32x2 h = {E::pack(acc[nt][mt][4 * vg] * r, acc[nt][mt][4 * vg + 1] * r),
                             E::pack(acc[nt][mt][4 * vg + 2] * r, acc[nt][mt][4 * vg + 3] * r)};
            u32x2 y;
            y[0] = E::pack(E::lo(wt[0]) * E::lo(h[0]), E::hi(wt[0]) * E::hi(h[0]));
            y[1] = E::pack(E::lo(wt[1]) * E::lo(h[1]), E::hi(wt[1]) * E::hi(h[1]));
            return y;
        }, pr.C);
        return;
    }
    store_via_lds([&](int mt, int nt, int vg) {
        u32x2 w;
        w[0] = E::pack(acc[nt][mt][4 * vg], acc[nt][mt][4 * vg + 1]);
        w[1] = E::pack(acc[nt][mt][4 * vg + 2], acc[nt][mt][4 * vg + 3]);
        return w;
    }, pr.C);
}

// registers the hand-scheduled tile uses besides its operands (see gen_gemm_loop.py)
#define LVX_GEMM_TILE_CLOBBERS "memory", "vcc", "scc", "m0", "v0", "v1", "v2", "v3", "v4", "v5", "v6", "v7", "v8", "v9", "v10", "v11", "v12", "v13", "v14", "v15", "v16", "v17", "v18", "v19", "v20", "v21", "v22", "v23", "v24", "v25", "v26", "v27", "v28", "v29", "v30", "v31", "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47", "v48", "v49", "v50", "v51", "v52", "v53", "v54", "v55", "v56", "v57", "v58", "v59", "v60", "v61", "v62", "v63", "v121", "v122", "v123", "v124", "v125", "v126", "v127", "v128", "v129", "v130", "v131", "v132", "v133", "v134", "v135", "v136", "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"

// One operand's part of a stage of gemm_tile_kernel: ROWS rows x 64 k in pieces of 1 KiB (what one load of a
// wave fills).
//   !TRANS (memory [row][k]): LDS row r at r * 128 B; its 16-byte chunk c (k = 8c .. 8c+7) sits at position
//       c ^ ((r >> 1) & 7): of 16 consecutive rows the eight even and the eight odd ones, which share
//       the 256 bytes of a pass over the banks pairwise, each land in eight different positions
//    TRANS (memory [k][row]): LDS k-row at k * ROWS * 2 B; its chunk q (rows 8q .. 8q+7) at q ^ ((k & 3) << 2)
constexpr int TK = 64;                 // contraction depth of one stage
template <bool TRANS, int ROWS>
struct TileOperand {
    static constexpr int BYTES = ROWS * TK * 2, PIECES = BYTES / 1024, LPR = ROWS / 8;
    // what lane `lane` fetches of piece `ch`: byte offset from row r0 (column r0) of the operand, clamped to
    // its last row, and the k position inside the stage
    __device__ __forceinline__ static uint32_t src(int ch, int lane, int r0, int R, int64_t ld, int& kpos) {
        if (!TRANS) {
            const int row = 8 * ch + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
            kpos = c * 8;
            return (uint32_t)(min(r0 + row, R - 1) - r0) * (uint32_t)ld * 2u + (uint32_t)c * 16u;
        }
        const int k = ch * (64 / LPR) + lane / LPR, q = (lane % LPR) ^ ((k & 3) << 2);
        kpos = k;
        return (uint32_t)k * (uint32_t)ld * 2u + (uint32_t)(min(r0 + q * 8, R - 8) - r0) * 2u;
    }
    // LDS byte offsets of a wave's operand reads, first 32-row tile j0: !TRANS per k-step (add tile * 4096),
    // TRANS per tile (add k-step * 32 * ROWS)
    __device__ __forceinline__ static void read_offsets(uint32_t (&rd)[4], int j0, int lane) {
        const int l32 = lane & 31, g = lane >> 5, r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            rd[i] = TRANS ? (uint32_t)((8 * g + r) * ROWS * 2 + 64 * ((j0 + i) ^ r) + (2 * u + (t >> 1)) * 16 + (t & 1) * 8)
                          : (uint32_t)(j0 * 4096 + l32 * 128 + (((2 * i + g) ^ ((l32 >> 1) & 7)) << 4));
    }
};

// The TM x TN tile of the projections and their gradients: four waves of 128 x TN / 2 (TM = 224: 224 x 64) in one
// generated statement (gen_gemm_loop.py), then the C tile, 16-bit in LDS by then, leaves as whole row segments -
// through the RMS norm where problem 0 has one (16 lanes hold a head's 128 columns of a row).
// Bound by the matrix pipe and the power it may draw: MFMAs alone on N(0, 1) data sustain 1800 TFLOP/s on the
// chip, this kernel 1341 (65536 x 4096 x 1024 twice, W [N][K]; 1215 with eight waves of 128 x 64 and stages
// of 32).  us before and after: that 905 -> 820; 12808 rows 183 -> 176; 2046 x 4096 x 4096 77 -> 60; the
// weight gradients, until then compiler-scheduled, 12808 rows 258 -> 168 and 6404 rows 134 -> 88.
template <bool A_T, bool B_T, int TN, bool F16, int TM>
__global__ __launch_bounds__(256, 1) void gemm_tile_kernel(const GemmParams p) {
    using E = Elt<F16>;
    static_assert(TM == 256 || (TM == 224 && TN == 256 && !A_T), "the tiles that are generated");
    constexpr int WM = TM == 256 ? 4 : 7, WN = TM == 256 ? TN / 64 : 2;
    using RA = TileOperand<A_T, TM>;
    using RB = TileOperand<B_T, TN>;
    constexpr int NSA = 3, NSB = TN == 256 ? 2 : 3, NLA = RA::PIECES / 4, NLB = RB::PIECES / 4, NL = NLA + NLB;
    __shared__ __attribute__((aligned(1024))) char lds[NSA * RA::BYTES + NSB * RB::BYTES];
    static_assert(sizeof(lds) >= TM * TN * 2, "the C tile takes the stages' place");

    fetch_kernargs<sizeof(GemmParams)>();
    const int wid = xcd_remap(blockIdx.x, p.total_wg);
    if (wid >= p.total_wg) return;
    uint32_t tn, prob;
    // the problems of an M tile side by side: they share an operand (K and V the visual states), which then
    // is read from HBM once
    const int tm = p.by_nprob.split(p.by_tiles_n.split(wid, tn), prob);
    const GemmProblem& pr = p.prob[prob];
    const int m0 = tm * TM, n0 = tn * TN;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wm = TM == 256 ? wave & 1 : 0, wn = TM == 256 ? wave >> 1 : wave;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    const int64_t lda = pr.lda[0], ldb = pr.ldb[0];
    const int st0 = (pr.K[0] + TK - 1) / TK, nst = st0 + (pr.nseg > 1 ? st0 : 0);      // both segments have one length
    const int tail = pr.K[0] % TK;

    // This wave's pieces of a stage: offsets from the tile's first row (column) of the operand.  In the last
    // stage, 16-byte pieces past the end of a contraction that is contiguous in memory are sent out of
    // the descriptor's range; where it is not contiguous the range itself ends with it.
    uint32_t voff[16], vtail[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        if (j >= NL) { voff[j] = vtail[j] = 0; continue; }
        int kpos;
        const int ch = wave + 4 * (j < NLA ? j : j - NLA);
        voff[j] = j < NLA ? RA::src(ch, lane, m0, p.M, lda, kpos) : RB::src(ch, lane, n0, p.N, ldb, kpos);
        vtail[j] = tail && kpos >= tail && !(j < NLA ? A_T : B_T) ? 0x80000000u : voff[j];
        if (nst == 1) voff[j] = vtail[j];
    }
    typedef __attribute__((ext_vector_type(4))) uint32_t srd_t;
    auto descriptor = [&](const uint16_t* base, int64_t ld, bool trans) {
        const uint64_t addr = (uint64_t)(uintptr_t)base;
        srd_t d;
        d[0] = uniform32((uint32_t)addr);
        d[1] = uniform32((uint32_t)(addr >> 32) & 0xffffu);
        d[2] = uniform32(trans ? (uint32_t)((uint64_t)pr.K[0] * (uint64_t)ld * 2u) : 0x7fffffffu);
        d[3] = 0x00020000u;
        return d;
    };
    auto a_base = [&](int i) { return pr.A[i] + (A_T ? (int64_t)m0 : (int64_t)m0 * lda); };
    auto b_base = [&](int i) { return pr.Bm[i] + (B_T ? (int64_t)n0 : (int64_t)n0 * ldb); };
    srd_t sa = descriptor(a_base(0), lda, A_T), sb = descriptor(b_base(0), ldb, B_T);
    const int second = pr.nseg > 1 ? 1 : 0;
    const uint64_t a1 = (uint64_t)uniform64((int64_t)(uintptr_t)a_base(second) & 0xffffffffffffll);
    const uint64_t b1 = (uint64_t)uniform64((int64_t)(uintptr_t)b_base(second) & 0xffffffffffffll);
    const uint32_t a_step = (uint32_t)(A_T ? lda * TK * 2 : TK * 2), b_step = (uint32_t)(B_T ? ldb * TK * 2 : TK * 2);

    uint32_t rda[4], rdb[4], ra[12], rb[12];
    RA::read_offsets(rda, WM * wm, lane);
    RB::read_offsets(rdb, WN * wn, lane);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
        ra[i] = lds0 + rda[i & 3] + (i >> 2) * RA::BYTES;
        rb[i] = lds0 + NSA * RA::BYTES + rdb[i & 3] + min(i >> 2, NSB - 1) * RB::BYTES;
    }
    // The C tile in LDS: 16-byte chunk c of row r at position c ^ (r mod chunks per row), its two 8-byte halves
    // exchanged in rows where bits 3 and 4 differ: the 8-byte writes of 32 rows and the 16-byte reads of
    // whole rows are both conflict-free.
    constexpr int CPR = TN / 8;
    const uint32_t ep = lds0 + (uint32_t)((128 * wm + l32) * (TN * 2) + (((4 * WN * wn) ^ (l32 & (CPR - 1))) << 4) +
                                          ((g ^ ((l32 >> 3) & 1) ^ (l32 >> 4)) << 3));
    uint32_t left = uniform32((uint32_t)nst), ahead = uniform32((uint32_t)(nst - 1)), soa = 0, sob = 0;
    uint32_t to_second = uniform32((uint32_t)(pr.nseg > 1 ? st0 : 0)), ahead_b = ahead, to_second_b = to_second;
#define LVX_GEMM_TILE_OPERANDS \
    : "+{v64}"(voff[0]), "+{v65}"(voff[1]), "+{v66}"(voff[2]), "+{v67}"(voff[3]), "+{v68}"(voff[4]), "+{v69}"(voff[5]), \
      "+{v70}"(voff[6]), "+{v71}"(voff[7]), "+{v72}"(voff[8]), "+{v73}"(voff[9]), "+{v74}"(voff[10]), "+{v75}"(voff[11]), \
      "+{v76}"(voff[12]), "+{v77}"(voff[13]), "+{v78}"(voff[14]), "+{v79}"(voff[15]), "+{s[40:43]}"(sa), "+{s[44:47]}"(sb), \
      "+{s51}"(left), "+{s52}"(ahead), "+{s53}"(soa), "+{s54}"(sob), "+{s55}"(to_second), "+{s60}"(ahead_b), "+{s61}"(to_second_b) \
    : "{v80}"(vtail[0]), "{v81}"(vtail[1]), "{v82}"(vtail[2]), "{v83}"(vtail[3]), "{v84}"(vtail[4]), "{v85}"(vtail[5]), \
      "{v86}"(vtail[6]), "{v87}"(vtail[7]), "{v88}"(vtail[8]), "{v89}"(vtail[9]), "{v90}"(vtail[10]), "{v91}"(vtail[11]), \
      "{v92}"(vtail[12]), "{v93}"(vtail[13]), "{v94}"(vtail[14]), "{v95}"(vtail[15]), "{v96}"(ra[0]), "{v97}"(ra[1]), \
      "{v98}"(ra[2]), "{v99}"(ra[3]), "{v100}"(ra[4]), "{v101}"(ra[5]), "{v102}"(ra[6]), "{v103}"(ra[7]), \
      "{v104}"(ra[8]), "{v105}"(ra[9]), "{v106}"(ra[10]), "{v107}"(ra[11]), "{v108}"(rb[0]), "{v109}"(rb[1]), \
      "{v110}"(rb[2]), "{v111}"(rb[3]), "{v112}"(rb[4]), "{v113}"(rb[5]), "{v114}"(rb[6]), "{v115}"(rb[7]), \
      "{v116}"(rb[8]), "{v117}"(rb[9]), "{v118}"(rb[10]), "{v119}"(rb[11]), "{v120}"(ep), \
      "{s48}"(uniform32(a_step)), "{s49}"(uniform32(b_step)), "{s50}"(uniform32(lds0 + (uint32_t)wave * 1024u)),  \
      "{s[56:57]}"(a1), "{s[58:59]}"(b1)                                                                         \
    : LVX_GEMM_TILE_CLOBBERS
    // one statement per layout, width and type; the text takes the instruction names from these macros
    if constexpr (!F16) {
#define LVX_GEMM_MFMA "v_mfma_f32_32x32x16_bf16"
#define LVX_GEMM_CVT "v_cvt_pk_bf16_f32"
        if constexpr (!A_T && !B_T && TN == 256 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pp_256_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && !B_T && TN == 128 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pp_128_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && B_T && TN == 256 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pt_256_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && B_T && TN == 128 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pt_128_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (A_T && B_T && TN == 256 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_tt_256_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (A_T && B_T && TN == 128 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_tt_128_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && B_T && TM == 224) {
            asm volatile(
#include "lvx_gemm_loop_pt_256_224.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && !B_T && TM == 224) {
            asm volatile(
#include "lvx_gemm_loop_pp_256_224.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
#undef LVX_GEMM_MFMA
#undef LVX_GEMM_CVT
    } else {
#define LVX_GEMM_MFMA "v_mfma_f32_32x32x16_f16"
#define LVX_GEMM_CVT "v_cvt_pk_f16_f32"
        if constexpr (!A_T && !B_T && TN == 256 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pp_256_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && !B_T && TN == 128 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pp_128_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && B_T && TN == 256 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pt_256_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && B_T && TN == 128 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_pt_128_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (A_T && B_T && TN == 256 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_tt_256_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (A_T && B_T && TN == 128 && TM == 256) {
            asm volatile(
#include "lvx_gemm_loop_tt_128_256.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && B_T && TM == 224) {
            asm volatile(
#include "lvx_gemm_loop_pt_256_224.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
        else if constexpr (!A_T && !B_T && TM == 224) {
            asm volatile(
#include "lvx_gemm_loop_pp_256_224.inc"
                LVX_GEMM_TILE_OPERANDS);
        }
#undef LVX_GEMM_MFMA
#undef LVX_GEMM_CVT
    }
    __syncthreads();

    uint16_t* const C = pr.C;
    const bool norm = p.norm_w && prob == 0;
    const int cc = tid % CPR, n = n0 + cc * 8;
    const u32x4 wt = norm && n < p.N ? *reinterpret_cast<const u32x4*>(p.norm_w + (n & 127)) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll 4
    for (int i = 0; i < TM * CPR / 256; ++i) {
        const int row = i * (256 / CPR) + tid / CPR, m = m0 + row;
        u32x4 val = *reinterpret_cast<const u32x4*>(lds + row * (TN * 2) + ((cc ^ (row & (CPR - 1))) << 4));
        if (((row >> 3) ^ (row >> 4)) & 1) val = u32x4{val[2], val[3], val[0], val[1]};
        const bool ok = m < p.M && n < p.N;
        if (norm) {
            // RMS norm over the head's 128 columns, 16 lanes (summed by shuffles, K and V of 12808 rows with it took 224
            // us; 221 so): y = rn(w * rn(x * r)), x the product as 16 bits
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                ss = fmaf(E::lo(val[j]), E::lo(val[j]), ss);
                ss = fmaf(E::hi(val[j]), E::hi(val[j]), ss);
            }
            ss = sum16(ss);
            const float r = rsqrtf(ss * (1.f / 128.f) + p.norm_eps);
            if (ok && p.rstd && (cc & 15) == 0) p.rstd[(int64_t)m * (p.N >> 7) + (n >> 7)] = r;
            if (ok && p.c_raw) __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(p.c_raw + (int64_t)m * pr.ldc + n));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t h = E::pack(E::lo(val[j]) * r, E::hi(val[j]) * r);
                val[j] = E::pack(E::lo(wt[j]) * E::lo(h), E::hi(wt[j]) * E::hi(h));
            }
        }
        // (a streaming store: nobody on this CU reads the tile again)
        if (ok) __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(C + (int64_t)m * pr.ldc + n));
    }
}

// The tiles of a launch and the divisors by what its work-group numbers are made of.
void fill_tiles(GemmParams& p, int TM, int TN) {
    p.tiles_m = (p.M + TM - 1) / TM;
    p.tiles_n = (p.N + TN - 1) / TN;
    p.total_wg = p.nprob * p.tiles_m * p.tiles_n;
    p.by_tiles_n = divisor(p.tiles_n);
    p.by_tiles_m = divisor(p.tiles_m);
    p.by_nprob = divisor(p.nprob);
}

template <int GM, int GN, int WM, int WN, int NS, bool F16>
hipError_t launch_cfg_t(const GemmParams& p, int grid, bool a_mcontig, bool b_ncontig, hipStream_t st) {
    if (!a_mcontig && !b_ncontig)
        return launch1((gemm_kernel<false, false, GM, GN, WM, WN, NS, F16>), dim3(grid), dim3(512), st, p);
    else if (!a_mcontig && b_ncontig)
        return launch1((gemm_kernel<false, true, GM, GN, WM, WN, NS, F16>), dim3(grid), dim3(512), st, p);
    else if (a_mcontig && !b_ncontig)
        return launch1((gemm_kernel<true, false, GM, GN, WM, WN, NS, F16>), dim3(grid), dim3(512), st, p);
    return launch1((gemm_kernel<true, true, GM, GN, WM, WN, NS, F16>), dim3(grid), dim3(512), st, p);
}

template <int GM, int GN, int WM, int WN, int NS>
hipError_t launch_cfg(GemmParams p, bool a_mcontig, bool b_ncontig, hipStream_t st) {
    fill_tiles(p, 32 * WM * GM, 32 * WN * GN);
    const int grid = ((p.total_wg + 7) / 8) * 8;
    if (p.f16) return launch_cfg_t<GM, GN, WM, WN, NS, true>(p, grid, a_mcontig, b_ncontig, st);
    return launch_cfg_t<GM, GN, WM, WN, NS, false>(p, grid, a_mcontig, b_ncontig, st);
}


template <int TN, bool F16, int TM = 256>
hipError_t launch_tile(GemmParams p, bool a_mcontig, bool b_ncontig, hipStream_t st) {
    fill_tiles(p, TM, TN);
    const dim3 grid((p.total_wg + 7) / 8 * 8);
    if (!a_mcontig && !b_ncontig) return launch1((gemm_tile_kernel<false, false, TN, F16, TM>), grid, dim3(256), st, p);
    if (!a_mcontig) return launch1((gemm_tile_kernel<false, true, TN, F16, TM>), grid, dim3(256), st, p);
    if constexpr (TM == 256) return launch1((gemm_tile_kernel<true, true, TN, F16, TM>), grid, dim3(256), st, p);
    return hipErrorInvalidValue;
}

// What gemm_tile_kernel takes: one contraction length for both segments (whole stages of it where
// there are two), offsets inside an operand below 2^32, and not the layout nothing uses.
bool gemm_tile_ok(const GemmParams& p, bool a_mcontig, bool b_ncontig) {
    const GemmProblem& pr = p.prob[0];
    if (a_mcontig && !b_ncontig) return false;
    if (pr.nseg > 1 && (pr.K[1] != pr.K[0] || pr.K[0] % TK)) return false;
    // (the descriptor of a row-major operand covers 2 GiB, the other kind ends with the contraction)
    const int64_t limit = (int64_t)1 << 32;
    const int64_t a_end = (a_mcontig ? (pr.K[0] + 2 * TK) * pr.lda[0] : 256 * pr.lda[0] + pr.K[0]) * 2;
    const int64_t b_end = (b_ncontig ? (pr.K[0] + 2 * TK) * pr.ldb[0] : 256 * pr.ldb[0] + pr.K[0]) * 2;
    return a_end < (a_mcontig ? limit : limit / 2) && b_end < (b_ncontig ? limit : limit / 2);
}

}  // namespace

// Work-group tile by shape.  C wider than 128 columns (projections, their gradients): a hand-scheduled tile of 256 x 256,
// 256 x 128 or 224 x 256 (gemm_tile).
// A narrow C: 256 x 128, four stages.
hipError_t launch_gemm(const GemmParams& p, bool a_mcontig, bool b_ncontig, hipStream_t st) {
    if (p.N % 8) return hipErrorInvalidValue;
    for (int i = 0; i < p.nprob; ++i) {
        const GemmProblem& pr = p.prob[i];
        // all problems and both contraction segments share the per-thread load offsets
        if (pr.lda[0] != p.prob[0].lda[0] || pr.ldb[0] != p.prob[0].ldb[0]) return hipErrorInvalidValue;
        if (pr.nseg > 1 && (pr.lda[1] != pr.lda[0] || pr.ldb[1] != pr.ldb[0])) return hipErrorInvalidValue;
    }
    if (p.N > 128 && gemm_tile_ok(p, a_mcontig, b_ncontig)) {
        switch (gemm_tile(p.M, p.N, p.nprob, cu_count(), !a_mcontig)) {
            case TILE_224_256: return p.f16 ? launch_tile<256, true, 224>(p, a_mcontig, b_ncontig, st) : launch_tile<256, false, 224>(p, a_mcontig, b_ncontig, st);
            case TILE_256_128: return p.f16 ? launch_tile<128, true>(p, a_mcontig, b_ncontig, st) : launch_tile<128, false>(p, a_mcontig, b_ncontig, st);
            default: return p.f16 ? launch_tile<256, true>(p, a_mcontig, b_ncontig, st) : launch_tile<256, false>(p, a_mcontig, b_ncontig, st);
        }
    }
    if (p.N > 128) return launch_cfg<2, 4, 4, 2, 4>(p, a_mcontig, b_ncontig, st);
    return launch_cfg<4, 2, 2, 2, 4>(p, a_mcontig, b_ncontig, st);
}

}  // namespace lvx

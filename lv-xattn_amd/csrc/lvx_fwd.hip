// Flash cross-attention forward for gfx950: one launch computes, for a window
// of text rows, O = softmax(scale * Q K^T) V (bf16) and the per-row natural-log
// LSE against the local K/V shard (or one key split of it).
//
// Mapping.  A work-group is 4 wavefronts.  Each wavefront owns 32 text rows of
// ONE q head; the 4 waves of a group cover the q heads that share a kv head
// (G = 4: four heads x 32 rows; G = 1: one head x 128 rows), so the K/V tile
// staged in LDS is read by the whole GQA group and nothing is expanded in HBM.
// (That is fwd_kernel, which heads of 16 and 32 run and few rows with a dense bias.  Head dimensions 128 and 64 run
// fwd_wide_kernel, in which a wavefront owns 64 rows, and few rows fwd_few_kernel; see there.)
//
// Per 64-key tile and wave (all MFMA are v_mfma_f32_32x32x16_bf16):
//   S^T[key, row]  = K_tile (A, from LDS)  x  Q^T (B, 32 VGPRs held for the whole kernel)
//   online softmax : a lane owns one text row (column of S^T) and 32 of the 64
//                    keys, so max/sum are in-register plus ONE exchange between
//                    the two lane halves; rescaling O is a per-lane scalar
//   O^T[d, row]   += V^T_tile (A, from LDS) x  P^T (B, straight from the S^T
//                    accumulators: register v of lane-half g is key
//                    8*(v/4)+4*g+(v%4); the V^T operand is fetched from the
//                    row-major V tile with the transposing LDS read, addressed
//                    in that same key order, so P never visits LDS and V is
//                    never transposed in memory)
// K and V tiles ([64 keys][128] bf16, 16 KiB each) go from global memory
// straight into LDS with global_load_lds_dwordx4, double-buffered: tile t+1 is
// in flight while tile t is consumed, one barrier per tile, no staging
// registers and no LDS stores.  That load writes 64 lanes x 16 bytes
// contiguously, so rows cannot be padded; instead the 16-byte chunk c of row r
// is kept at position c ^ f(r), f(r) = ((r & 3) << 2) | ((r >> 2) & 3): the 16
// rows a 16-byte operand read of K touches land in 16 different positions, and
// the 4 rows a transposing read of V touches land in 4 different 64-byte
// groups - both conflict-free.  Loads past the end of the key range are
// clamped to its last row (those keys are masked out of S).
#include <type_traits>

#include "lvx_common.hpp"
#include "lvx_fold.hpp"
#include "lvx_kernels.hpp"

namespace lvx {

namespace {

constexpr int D = 128;
constexpr int BN = 64;        // keys per tile
constexpr int TILE_BYTES = BN * D * 2;
constexpr int BIG = 0x3fffffff;
constexpr float RESCALE_LOG2 = 8.f;
constexpr float LOG2E_F = 1.4426950408889634f, LN2_F = 0.6931471805599453f;

// LSE of a row whose sum of exponentials is not positive: -inf where it saw no key (0).  A NaN among its scores makes the
// sum NaN; a part of a launch with key splits then says NaN, so that the fold does not take it for a part that saw
// nothing and give the result without it.
__device__ __forceinline__ float no_lse(const FwdParams& p, float sum) { return (p.nsplit > 1 ? sum : 0.f) - INFINITY; }

// What a row that sees nothing has for Q (see fwd_wide_kernel).
__device__ const uint16_t zero_row[D] __attribute__((aligned(16))) = {};

// BIAS: a dense fp32 bias is added to scale * S before the softmax; the scores are
// then carried in log2 units (S*c + bias*log2e) instead of raw.
// DH: head dimension, 16, 32, 64 or 128.  The LDS tiles keep their 256-byte rows and chunk
// permutation whatever DH is: below 128 only the first DH / 8 chunks of a row hold data (the
// lanes that would load the others repeat a chunk of the same row), and the k-steps of S^T and
// the 32-wide blocks of O^T past DH do not exist.  With 16 the one block of O^T is half real:
// its upper 16 rows are products with those repeated chunks and are never stored.
template <int DH, bool MASKED, bool BIAS, bool F16>
__global__ __launch_bounds__(256, 2) void fwd_kernel(const FwdParams p) {
    using E = Elt<F16>;
    static_assert(DH == 16 || DH == 32 || DH == 64 || DH == 128, "head dimension");
    constexpr int NKK = DH / 16, NDT = DH >= 32 ? DH / 32 : 1;
    __shared__ __attribute__((aligned(1024))) char kv_lds[2][2][TILE_BYTES];   // [buffer][K, V]
    __shared__ int red[4][4];

    fetch_kernargs<sizeof(FwdParams)>();
    const int wid = xcd_remap(blockIdx.x, p.total_wg);
    if (wid >= p.total_wg) return;
    uint32_t tile, split, b;
    const uint32_t t1 = p.by_row_tiles.split(wid, tile), t2 = p.by_splits.split(t1, split);
    // samples vary faster than head groups: every XCD (a contiguous range of ids) then gets
    // work-groups of all samples, and ragged samples do not leave some XCDs idle early
    const uint32_t hg = p.by_B.split(t2, b);

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    // HG is 1, 2 or 4: the wave's head of the group and its row sub-tile
    const int wave_head = wave & (p.HG - 1), wave_rows = wave >> (p.HG >> 1);
    const int h = hg * p.HG + wave_head;
    uint32_t of_group;
    const int hk = p.by_G.split(h, of_group);
    const int row = p.row_begin + (tile * p.RS + wave_rows) * 32 + l32;
    const bool row_ok = row < p.row_end;

    int kv_len = p.Lkv;
    if (p.kv_len) kv_len = min(p.kv_len[b], p.Lkv);
    const int kv_lo = split * p.split_len;
    const int kv_hi = min(kv_len, kv_lo + p.split_len);

    // this lane's visible key interval
    int my_s = kv_lo, my_e = kv_hi;
    if (MASKED) {
        if (row_ok) {
            my_s = max(kv_lo, p.kv_start[(int64_t)b * p.Lq + row]);
            my_e = min(kv_hi, p.kv_end[(int64_t)b * p.Lq + row]);
        } else {
            my_e = my_s;
        }
    }
    if (my_e <= my_s) { my_s = BIG; my_e = 0; }

    // work-group key range: [lo, hi) covers every non-empty row; tiles inside
    // [in_lo, in_hi) are visible to every row and need no masking
    int lo = my_s, hi = my_e, in_lo = my_s, in_hi = my_e;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        lo = min(lo, __shfl_xor(lo, off));
        hi = max(hi, __shfl_xor(hi, off));
        in_lo = max(in_lo, __shfl_xor(in_lo, off));
        in_hi = min(in_hi, __shfl_xor(in_hi, off));
    }
    if (lane == 0) { red[wave][0] = lo; red[wave][1] = hi; red[wave][2] = in_lo; red[wave][3] = in_hi; }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        lo = min(lo, red[w][0]);
        hi = max(hi, red[w][1]);
        in_lo = max(in_lo, red[w][2]);
        in_hi = min(in_hi, red[w][3]);
    }
    // the same in every lane of the work-group: keep them in scalar registers
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    in_lo = __builtin_amdgcn_readfirstlane(in_lo);
    in_hi = __builtin_amdgcn_readfirstlane(in_hi);

    // Q^T as B operand, resident for the whole kernel
    bf16x8 qreg[NKK];
    {
        const uint16_t* qp = p.q + b * p.qs.b + h * p.qs.h + (int64_t)row * p.qs.s + g * 8;
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) qreg[kk] = as_bf16x8(ldg16(qp + kk * 16, row_ok));
    }

    const char* kbase = reinterpret_cast<const char*>(p.k + b * p.ks.b + hk * p.ks.h);
    const char* vbase = reinterpret_cast<const char*>(p.v + b * p.vs.b + hk * p.vs.h);
    const uint32_t krow_b = (uint32_t)p.ks.s * 2u, vrow_b = (uint32_t)p.vs.s * 2u;   // bytes per key row

    // global -> LDS: wave w moves the 1 KiB chunks w, w+4, w+8, w+12 (4 rows each)
    // of the K tile and of the V tile; lane i fills position i & 15 of row i >> 4.
    const int wave_u = wave;
    const int ld_r = lane >> 4;
    const uint32_t ld_c = (uint32_t)(((lane & 15) ^ ((ld_r << 2) | wave_u)) & (DH / 8 - 1)) * 16u;   // chunk this lane fetches
    const uint32_t lds0 = (uint32_t)(uintptr_t)&kv_lds[0][0][0];
    auto issue = [&](int kv0, int buf) {
        const char* kb = kbase + (int64_t)kv0 * krow_b;
        const char* vb = vbase + (int64_t)kv0 * vrow_b;
        const uint32_t slot = lds0 + (uint32_t)buf * (2 * TILE_BYTES) + (uint32_t)wave_u * 1024u;
        const int last = kv_hi - 1 - kv0;          // rows past `last` repeat it
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t r = (uint32_t)min(4 * (wave_u + 4 * j) + ld_r, last);
            dma16(kb, r * krow_b + ld_c, slot + j * 4096);
            dma16(vb, r * vrow_b + ld_c, slot + TILE_BYTES + j * 4096);
        }
    };

    // LDS -> operands.  K rows (A of S^T): 16 bytes at row * 256 + ((2 kk + g) ^ f(row)) * 16.
    const int f_row = ((l32 & 3) << 2) | ((l32 >> 2) & 3);
    const uint32_t k_rd = (uint32_t)(l32 * 256), k_h = (uint32_t)((g ^ f_row) << 4);
    // V^T (A of O^T += V^T P^T), keys in accumulator order: first half rows 16 j + 4 g + r,
    // second half 8 rows further down, whose f differs in bit 1.
    uint32_t v_rd[4][2];
    {
        const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
        const int low = (2 * u + (t >> 1)) ^ g;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            v_rd[dt][0] = (uint32_t)((4 * g + r) * 256 + (4 * (dt ^ r) + low) * 16 + (t & 1) * 8);
            v_rd[dt][1] = (uint32_t)((4 * g + r + 8) * 256 + (4 * (dt ^ r) + (low ^ 2)) * 16 + (t & 1) * 8);
        }
    }

    f32x16 acc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[dt][v] = 0.f;
    float m_i = -INFINITY, l_i = 0.f;
    const float c = p.scale_log2e;
    const float cc = BIAS ? 1.f : c;              // factor from the carried scores to log2 units
    const float* brow = nullptr;                  // this lane's row of the bias
    if (BIAS) brow = p.bias + b * p.bias_b + h * p.bias_h + (int64_t)min(row, p.row_end - 1) * p.bias_r;
    // The bias of a tile: register group vg of lane-half g holds keys kv0 + 8 vg + 4 g + 0..3, the second four 32 keys
    // further; groups past the end re-read the last one (those keys are masked).  A tile's values are requested
    // during the tile before, between the loads of its own K and V and those of the next.  (Requested where they are
    // used, behind the loads of the next tile, they were waited for together with those: 1024 rows x 16 heads x 4096
    // keys forward and backward 268 us, so 255.)  The request is assembly,
    // so the compiler does not know of the wait: nothing may touch the registers before it.
    // What is in flight is not waited for by these waits alone.  The compiler, which sees none of them, waits for Q in front
    // of every tile's first MFMA, and with it for the tile requested just before.  Made to wait for Q once in front of
    // the loop, the kernel takes 120 us instead of 151 where work-groups are few (1024 rows x 16 heads x 4096 keys in one
    // range; in the ranges that are chosen nothing), but more where they fill the chip, out of step and with the bias no longer
    // shared in the L2 (4096 x 32 heads x 6404 509 -> 520; heads of 64 396 -> 423, of 32 404 -> 435), and the
    // forward and backward above 247 -> 251.
    u32x4 bq[8];
    const int last_k = (p.Lkv - 1) & ~3;
    auto request_bias = [&](int kv0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float* at = brow + min(kv0 + 8 * (i & 3) + 4 * g + 32 * (i >> 2), last_k);
            asm volatile("global_load_dwordx4 %0, %1, off" : "+v"(bq[i]) : "v"(at) : "memory");
            __builtin_amdgcn_sched_barrier(0);      // one address at a time
        }
    };

    const int t_begin = (hi > lo) ? lo / BN : 0;
    const int t_end = (hi > lo) ? (hi + BN - 1) / BN : 0;
    if (t_end > t_begin) {
        issue(t_begin * BN, 0);
        if (BIAS) {
#pragma unroll
            for (int i = 0; i < 8; ++i) bq[i] = u32x4{0u, 0u, 0u, 0u};
            request_bias(t_begin * BN);
        }
    }

    for (int t = t_begin; t < t_end; ++t) {
        const int kv0 = t * BN;
        const int buf = (t - t_begin) & 1;
        const char* Ks = kv_lds[buf][0];
        const char* Vs = kv_lds[buf][1];

        // tile t has landed (this wave's part: vmcnt; everyone's: barrier); the
        // barrier also says every wave is done reading tile t-1, whose buffer
        // the loads of tile t+1 may now overwrite
        if (BIAS) wait_vmcnt<8>();          // the tile's bias, requested after it, may be on its way
        else wait_vmcnt<0>();
        lds_barrier();
        if (t + 1 < t_end) issue(kv0 + BN, buf ^ 1);

        // S^T = K Q^T : rows = keys (two 32-key sub-tiles), cols = text rows.
        // All 16 K operands are requested before the first MFMA, so the LDS
        // latency is paid once per tile and not once per k-step.
        bf16x8 ka[NKK][2];
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
            const char* kp = Ks + k_rd + ((uint32_t)(kk * 32) ^ k_h);
            ka[kk][0] = *reinterpret_cast<const bf16x8*>(kp);
            ka[kk][1] = *reinterpret_cast<const bf16x8*>(kp + 32 * 256);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x16 s0, s1;
#pragma unroll
        for (int v = 0; v < 16; ++v) { s0[v] = 0.f; s1[v] = 0.f; }
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
            s0 = E::mfma(ka[kk][0], qreg[kk], s0);
            s1 = E::mfma(ka[kk][1], qreg[kk], s1);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (BIAS) {
            if (t + 1 < t_end) wait_vmcnt<8>();         // all but the loads of the next tile (none by now, see above)
            else wait_vmcnt<0>();
#pragma unroll
            for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(bq[i]));
#pragma unroll
            for (int vg = 0; vg < 4; ++vg)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    s0[4 * vg + r] = fmaf(s0[4 * vg + r], c, __uint_as_float(bq[vg][r]) * LOG2E_F);
                    s1[4 * vg + r] = fmaf(s1[4 * vg + r], c, __uint_as_float(bq[4 + vg][r]) * LOG2E_F);
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        // V^T operands of this tile: requested now, they land during the softmax
        u32x2 va[NDT][4][2];
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                va[dt][j][0] = lds_read_tr16(reinterpret_cast<const uint16_t*>(Vs + v_rd[dt][0] + j * 4096));
                va[dt][j][1] = lds_read_tr16(reinterpret_cast<const uint16_t*>(Vs + v_rd[dt][1] + j * 4096));
            }
        __builtin_amdgcn_sched_barrier(0);

        if (kv0 < in_lo || kv0 + BN > in_hi) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int kv = kv0 + acc_row(v, g);
                if (kv < my_s || kv >= my_e) s0[v] = -INFINITY;
                if (kv + 32 < my_s || kv + 32 >= my_e) s1[v] = -INFINITY;
            }
        }

        mfma_settle(s0, s1);
        float mx = max3(s0[0], s1[0], s0[1]);
        mx = max3(mx, s1[1], s0[2]);
#pragma unroll
        for (int v = 3; v < 16; v += 1) mx = max3(mx, s1[v - 1], s0[v]);
        mx = fmaxf(mx, s1[15]);
        {   // other half of the wave holds the other 32 keys of the same text row
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = max3(__uint_as_float(sw[0]), __uint_as_float(sw[1]), m_i);
        }
        // Lazy rescale: the reference point m_i of a row only moves when the row
        // maximum has grown by more than 2^RESCALE_LOG2 since it was set, so P may
        // reach 2^RESCALE_LOG2 instead of 1 (harmless in fp32 / bf16) and the
        // rescale of O happens a few times per row instead of almost every tile.
        const float mcand = mx * cc;                      // mx >= m_i
        const float m_ic = m_i * cc;
        const bool move = (mx != -INFINITY) && !(mcand - m_ic <= RESCALE_LOG2);
        const float alpha = move ? __builtin_amdgcn_exp2f(m_ic - mcand) : 1.f;
        if (move) m_i = mx;
        const float mc = (m_i == -INFINITY) ? 0.f : m_i * cc;

        // P^T as B operand: k-step j covers keys 16j..16j+15 of the tile.  The row
        // sum is taken in fp32 before the rounding to bf16 (summing the rounded
        // values would put the LSE off by up to a bf16 ulp of the largest term).
        bf16x8 pb[4];
        float rs0 = 0.f, rs1 = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            u32x4 u0, u1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int v = 8 * j + 2 * e;
                const float a0 = __builtin_amdgcn_exp2f(fmaf(s0[v], cc, -mc)), a1 = __builtin_amdgcn_exp2f(fmaf(s0[v + 1], cc, -mc));
                const float b0 = __builtin_amdgcn_exp2f(fmaf(s1[v], cc, -mc)), b1 = __builtin_amdgcn_exp2f(fmaf(s1[v + 1], cc, -mc));
                rs0 += a0 + a1;
                rs1 += b0 + b1;
                u0[e] = E::pack(a0, a1);
                u1[e] = E::pack(b0, b1);
            }
            pb[j] = as_bf16x8(u0);
            pb[2 + j] = as_bf16x8(u1);
        }
        l_i = l_i * alpha + (rs0 + rs1);

        if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {   // the running max moved for some row
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[dt][v] *= alpha;
        }

        // O^T += V^T P^T
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32x4 a = {va[dt][j][0][0], va[dt][j][0][1], va[dt][j][1][0], va[dt][j][1][1]};
                acc[dt] = E::mfma(as_bf16x8(a), pb[j], acc[dt]);
                // registers that the first half of V^T has left take the next tile's bias
                if (BIAS && dt == (NDT - 1) / 2 && j == 3) request_bias(min(kv0 + BN, last_k));
            }
    }

    if (BIAS && t_end > t_begin) {      // the last request has to land before its registers serve anything else
        wait_vmcnt<0>();
#pragma unroll
        for (int i = 0; i < 8; ++i) asm volatile("" ::"v"(bq[i]));
    }
    // epilogue: the two lane halves hold partial row sums of the same row
    const float l_tot = l_i + __shfl_xor(l_i, 32);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if (row_ok) {
        const int64_t at = split * p.o_split_stride + b * p.os.b + h * p.os.h + (int64_t)row * p.os.s;
        uint16_t* op = p.o + at;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int vg = 0; vg < 4; ++vg) {
                if (dt * 32 + 8 * vg + 4 * g >= DH) continue;      // only with DH = 16
                if (p.o_f32) {
                    const f32x4 x = {acc[dt][4 * vg] * inv, acc[dt][4 * vg + 1] * inv, acc[dt][4 * vg + 2] * inv, acc[dt][4 * vg + 3] * inv};
                    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.o) + at + dt * 32 + 8 * vg + 4 * g) = x;
                    continue;
                }
                u32x2 w;
                w[0] = E::pack(acc[dt][4 * vg] * inv, acc[dt][4 * vg + 1] * inv);
                w[1] = E::pack(acc[dt][4 * vg + 2] * inv, acc[dt][4 * vg + 3] * inv);
                *reinterpret_cast<u32x2*>(op + dt * 32 + 8 * vg + 4 * g) = w;
            }
        if (g == 0) {
            const float lse = l_tot > 0.f ? m_i * (BIAS ? LN2_F : p.scale) + __logf(l_tot) : no_lse(p, l_tot);
            p.lse[split * p.lse_split_stride + ((int64_t)b * p.Hq + h) * p.lse_bh_stride + row] = lse;
        }
    }
}

// registers the wide loop uses besides its operands (see gen_fwd_loop_wide.py), heads of 128 and of 64
#define LVX_FWD_WIDE_CLOBBERS_128 "v132", "v133", "v134", "v135", "v136", "v137", "v138", "v139", "v140", "v141", "v142", "v143", "v144", "v145", "v146", "v147", "v148", "v149", "v150", "v151", "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159", "v160", "v161", "v162", "v163", "v164", "v165", "v166", "v167", "v168", "v169", "v170", "v171", "v172", "v173", "v174", "v175", "v176", "v177", "v178", "v179", "v180", "v181", "v182", "v183", "v184", "v185", "v186", "v187", "v188", "v189", "v190", "v191", "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", "v233", "v234", "v235", "v236", "v237", "v238", "v239", "v240", "v241", "v242", "v243", "v244", "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191"
#define LVX_FWD_WIDE_CLOBBERS_64 "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47", "v48", "v49", "v50", "v51", "v52", "v53", "v54", "v55", "v56", "v57", "v58", "v59", "v60", "v61", "v62", "v63", "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127", "v132", "v133", "v134", "v135", "v136", "v137", "v138", "v139", "v140", "v141", "v142", "v143", "v144", "v145", "v146", "v147", "v148", "v149", "v150", "v151", "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159", "v160", "v161", "v162", "v163", "v164", "v165", "v166", "v167", "v168", "v169", "v170", "v171", "v172", "v173", "v174", "v175", "v176", "v177", "v178", "v179", "v180", "v181", "v182", "v183", "v184", "v185", "v186", "v187", "v188", "v189", "v190", "v191", "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", "v204", "v205", "v206", "v207", "v212", "v213", "v214", "v215", "v218", "v219", "v222", "v223", "v233", "v234", "v235", "v236", "v237", "v238", "v239", "v240", "v241", "v242", "v243", "v244", "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175"
#define LVX_FWD_WIDE_CLOBBERS_S "memory", "vcc", "scc", "m0", "s52", "s53", "s54", "s55", "s56", "s58", "s59", "s60", "s61", "s70", "s71"

// Folds a share of what the launch before left in parts: the rows of a query block that has been computed, in the launch that
// computes the next, where fold_rides says so.  A launch of its own for it takes 6 us of the 35 that a round of 256 rows x 6404
// keys does.  Here it stands in front of the work-group's own loads, all parts of two chunks of a row in flight per thread, and
// takes 5 (a launch that folds 37.7 us, one that does not 33.2): 21 MB on their way back from the memory side, where the end of
// a launch leaves them.  Sixteen such rounds 593 -> 565 us.
// Heads go slowest over the work-groups, as in the launch that wrote the parts.
template <int DH, bool F16, int CHAINS>
__device__ __forceinline__ void fold_before(const FwdFoldParams& p, uint32_t wid) {
    using E = Elt<F16>;
    constexpr int SH = DH == 128 ? 4 : 3;
    const FwdFold& f = p.fold;
    const uint32_t n = (uint32_t)(p.B * p.Hq * f.rows) << SH, end = min((wid + 1) * f.per_wg, n);
    const int64_t l_stride = (int64_t)p.B * p.Hq * f.rows, stride = l_stride * DH;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (uint32_t at = wid * f.per_wg + threadIdx.x; at < end; at += 512) {
        uint32_t row[2], b[2], h[2];
        const int chunk = (int)(at & ((1 << SH) - 1));
        float l[2][CHAINS][FOLD_BATCH], la[2];
        u32x4 u[2][CHAINS][FOLD_BATCH], ua[2];
        RowFold sum[2][CHAINS];
        for (int k0 = 0; k0 < f.nparts; k0 += CHAINS * FOLD_BATCH) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const uint32_t r = (at + 256 * c < end ? at + 256 * c : at) >> SH;      // (past the share: the first again, dropped below)
                h[c] = p.by_B.split(f.by_rows.split(r, row[c]), b[c]);
                const int64_t bh = (int64_t)b[c] * p.Hq + h[c];
                const uint16_t* const op = f.part + (bh * f.rows + row[c]) * DH + chunk * 8;
                const float* const lp = f.l_part + bh * f.rows + row[c];
#pragma unroll
                for (int x = 0; x < CHAINS; ++x)
#pragma unroll
                    for (int k = 0; k < FOLD_BATCH; ++k) {
                        const int part = k0 + x + k * CHAINS, some = min(part, f.nparts - 1);
                        l[c][x][k] = lp[some * l_stride];
                        u[c][x][k] = *reinterpret_cast<const u32x4*>(op + some * stride);
                    }
                la[c] = -INFINITY;
                ua[c] = zero;
                if (f.acc) {
                    la[c] = f.l_acc[bh * p.Lq + f.row_begin + row[c]];
                    ua[c] = *reinterpret_cast<const u32x4*>(f.acc + b[c] * f.as.b + h[c] * f.as.h + row[c] * f.as.s + chunk * 8);
                }
            }
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int x = 0; x < CHAINS; ++x) {
#pragma unroll
                    for (int k = 0; k < FOLD_BATCH; ++k)
                        if (k0 + x + k * CHAINS >= f.nparts) l[c][x][k] = -INFINITY;
                    sum[c][x].add(l[c][x], [&](int k, float (&v)[8]) { unpack8<E>(u[c][x][k], v); });
                }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (at + 256 * c >= end) break;
            if (f.acc) {
                const float only[FOLD_BATCH] = {la[c], -INFINITY, -INFINITY, -INFINITY};
                sum[c][0].add(only, [&](int k, float (&v)[8]) { unpack8<E>(k ? zero : ua[c], v); });
            }
            if constexpr (CHAINS == 2) sum[c][0].join(sum[c][1]);
            *reinterpret_cast<u32x4*>(f.o + b[c] * f.os.b + h[c] * f.os.h + row[c] * f.os.s + chunk * 8) = sum[c][0].template result<E>();
            if (chunk == 0) f.l[((int64_t)b[c] * p.Hq + h[c]) * p.Lq + f.row_begin + row[c]] = sum[c][0].lse();
        }
    }
}

// The wide form (head dimensions 128 and 64, both element types, any mask): a wave
// owns two blocks of 32 rows of its head and has its SIMD to itself (one work-group per CU, 512
// registers per lane), so that every K / V operand read from LDS feeds two MFMAs: half the LDS reads
// and half the global -> LDS bytes per MFMA of fwd_kernel.  All key tiles of the work-group - whole,
// partial, masked, one or many - run in one hand-scheduled statement (gen_fwd_loop_wide.py): a tile in
// compiler-scheduled code costs a wave of 512 registers 4 - 7 us, one in the loop 1.1 - 1.6.
// Bound by the matrix pipe: 4096 rows x 32 heads x 6404 keys (0.43 TFLOP) takes 354 us, 1215 TFLOP/s,
// where fwd_kernel takes 429; 2 x 3000 rows with image intervals 332 -> 261; 2 x 1023 rows 202 -> 182;
// heads of 64, 2048 rows 145 -> 118 (half the MFMAs for the same softmax: bound by the VALU).
// What a work-group takes besides its tiles, which is all that launches of few tiles have to save: the first scores are
// formed 3.3 us after its first instruction (4.9 when the arguments came line by line, the numbers of the work-group
// from four integer divisions, and all loads behind 28 address computations with Q^T going through VGPRs), and 2.1 us
// pass behind the last tile.  One tile: 6.9 us from the first instruction to the last (8.7); sixteen launches of 256 rows
// x 6404 keys with their folds 661 -> 611, 2 x 300 rows eight times 574 -> 556.
//
// LDS tiles: row r of a K or V tile has 2 DH bytes; its 16-byte chunk c sits at position c ^ f(r).
//   DH = 128: f(r) = ((r & 3) << 2) | ((r >> 2) & 3), as in fwd_kernel
//   DH = 64 : two rows share the 256 bytes of a pass over the banks, and f(r) = ((r >> 1 & 1) << 2) |
//             ((r >> 2) & 3): the eight even and the eight odd rows of sixteen consecutive ones land
//             in eight different positions each, and of the four rows of a transposing read those of
//             like parity in different 64-byte halves
// FOLD: the launch also folds the parts of the one before it (a test at run time costs every launch 0.2 %).
// BIAS: the bias is added in the loop (see gen_fwd_loop_wide.py); intervals per row are optional then.  1024 rows x 16 heads x 4096
// keys, with the fold of four ranges 61.6 us in fwd_kernel -> 53.7, heads of 64 50.1 -> 40.1, 1024 x 32 x 6404 152 -> 130.  Without the
// bias's loads it would be 5 - 6 us less, without K's and V's as well 10; heads dealt to the XCDs side by side, so that they share
// a bias in L2, and more or fewer of its loads in the S phase change nothing (within 1 %).
template <int DH, bool MASKED, bool F16, bool FOLD, bool BIAS = false>
__global__ __launch_bounds__(256, 1) void fwd_wide_kernel(const std::conditional_t<FOLD, FwdFoldParams, FwdParams> p) {
    using E = Elt<F16>;
    static_assert(DH == 128 || DH == 64, "head dimension");
    constexpr int NKK = DH / 16, NDT = DH / 32, NLD = DH / 32;
    constexpr int ROWB = 2 * DH, TB = BN * ROWB, CPR = DH / 8;      // bytes per tile row and tile, chunks per row
    constexpr int RPL = 64 / CPR;                                   // tile rows one load of a wave fills
    constexpr int EP16 = ROWB + 16, EP32 = 4 * DH + 16;             // row strides of the tile that O leaves through
    constexpr int EPB = 64 * EP16;                                  // its bytes per wave (32 rows of floats fit too)
    static_assert(32 * EP32 <= EPB);
    constexpr int BIAS_BLOCK = 4 * 256 + 16, BIAS_TILE = 16 * BIAS_BLOCK;   // four rows of 64 floats, padded; 64 rows: a wave's tile
    __shared__ __attribute__((aligned(1024))) char kv_lds[4 * EPB + (BIAS ? 4 * BIAS_TILE : 0)];    // 4 TB: [buffer][K, V]; then O
    __shared__ int red[4][4];

    fetch_kernargs<sizeof(p)>();
    const int wid = xcd_remap(blockIdx.x, p.total_wg);
    if (wid >= p.total_wg) return;
    if constexpr (FOLD) {
        if (p.fold.chains == 2) fold_before<DH, F16, 2>(p, wid);
        else fold_before<DH, F16, 1>(p, wid);
    }
    uint32_t tile, split, b;
    const uint32_t t1 = p.by_row_tiles.split(wid, tile), t2 = p.by_splits.split(t1, split);
    // samples vary faster than head groups: every XCD (a contiguous range of ids) then gets
    // work-groups of all samples, and ragged samples do not leave some XCDs idle early
    const uint32_t hg = p.by_B.split(t2, b);

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int h = hg * p.HG + (wave & (p.HG - 1));       // HG is 1, 2 or 4, and RS = 4 / HG
    const int hk = p.by_head_groups.quotient(hg);
    const int row0 = p.row_begin + (tile * p.RS + (wave >> (p.HG >> 1))) * 64;      // this wave's first row

    int kv_len = p.Lkv;
    if (p.kv_len) kv_len = min(p.kv_len[b], p.Lkv);
    const int kv_lo = split * p.split_len;
    const int kv_hi = min(kv_len, kv_lo + p.split_len);

    // visible key interval of this lane's two rows.  Rows past the window and rows that see nothing
    // are let see everything, so that they do not make whole tiles take the element mask.  The former have the
    // window's last Q and are never stored: their scores are a lane's own, and if one moves its reference the wave rescales once
    // more.  The latter have a Q of zeros and are stored as zeros, which 0 times what a Q of infinities or NaN gives would
    // not be.
    int my_s[2] = {kv_lo, kv_lo}, my_e[2] = {kv_hi, kv_hi};
    bool empty[2] = {kv_hi <= kv_lo, kv_hi <= kv_lo};
    int lo = kv_lo, hi = kv_hi, in_lo = kv_lo, in_hi = kv_hi;
    if (MASKED && (!BIAS || p.kv_start)) {
        lo = BIG; hi = 0; in_lo = 0; in_hi = BIG;
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const int row = row0 + 32 * blk + l32;
            if (row < p.row_end) {
                my_s[blk] = max(kv_lo, p.kv_start[(int64_t)b * p.Lq + row]);
                my_e[blk] = min(kv_hi, p.kv_end[(int64_t)b * p.Lq + row]);
                empty[blk] = my_e[blk] <= my_s[blk];
                if (!empty[blk]) {
                    lo = min(lo, my_s[blk]);
                    hi = max(hi, my_e[blk]);
                    in_lo = max(in_lo, my_s[blk]);
                    in_hi = min(in_hi, my_e[blk]);
                }
            }
            if (row >= p.row_end || empty[blk]) { my_s[blk] = 0; my_e[blk] = BIG; }
        }
        // work-group key range: [lo, hi) covers every row, tiles inside [in_lo, in_hi) are visible to
        // every row and need no masking
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            lo = min(lo, __shfl_xor(lo, off));
            hi = max(hi, __shfl_xor(hi, off));
            in_lo = max(in_lo, __shfl_xor(in_lo, off));
            in_hi = min(in_hi, __shfl_xor(in_hi, off));
        }
        if (lane == 0) { red[wave][0] = lo; red[wave][1] = hi; red[wave][2] = in_lo; red[wave][3] = in_hi; }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            lo = min(lo, red[w][0]);
            hi = max(hi, red[w][1]);
            in_lo = max(in_lo, red[w][2]);
            in_hi = min(in_hi, red[w][3]);
        }
        lo = uniform32(lo); hi = uniform32(hi); in_lo = uniform32(in_lo); in_hi = uniform32(in_hi);
    }

    const int tile0 = hi > lo ? lo / BN : 0;
    const int n = uniform32(hi > lo ? (hi + BN - 1) / BN - tile0 : 0);     // key tiles of the work-group
    f32x16 acc[2][NDT];
    float m_i[2] = {-INFINITY, -INFINITY}, l_i[2] = {0.f, 0.f};
    if (n > 0) {
        const int kv0 = tile0 * BN;
        const uint32_t krow_b = (uint32_t)p.ks.s * 2u, vrow_b = (uint32_t)p.vs.s * 2u;   // bytes per key row
        const char* kp = uniform_ptr(reinterpret_cast<const char*>(p.k + b * p.ks.b + hk * p.ks.h) + (int64_t)kv0 * krow_b);
        const char* vp = uniform_ptr(reinterpret_cast<const char*>(p.v + b * p.vs.b + hk * p.vs.h) + (int64_t)kv0 * vrow_b);
        const uint32_t lds0 = (uint32_t)(uintptr_t)&kv_lds[0];
        const uint32_t lds_w = lds0 + (uint32_t)wave * 1024u;

        // global -> LDS: wave w fills the 1 KiB pieces w, w + 4, .. of a tile; lane i of a load fills
        // position i % CPR of row i / CPR of its piece.  Loads past the last key repeat its row
        // (those keys are masked out of S).
        const int ld_r = RPL * wave + lane / CPR;
        const uint32_t ld_c = (uint32_t)((lane % CPR) ^ (DH == 128 ? (((lane >> 4) << 2) | wave)
                                                                   : ((((lane >> 4) & 1) << 2) | ((2 * wave + (lane >> 5)) & 3)))) * 16u;
        const int last = hi - 1 - (kv0 + (n - 1) * BN);      // last row of the key range in the last tile
        auto piece_off = [&](int j, uint32_t rowb) {         // in the first tile, which may be the last
            const int r = ld_r + 4 * RPL * j;
            return (uint32_t)(n == 1 ? min(r, last) : r) * rowb + ld_c;
        };
        uint32_t dok[NLD], dov[NLD];
#pragma unroll
        for (int j = 0; j < NLD; ++j) { dok[j] = piece_off(j, krow_b); dov[j] = piece_off(j, vrow_b); }

        // Q^T as B operand: this lane's 16 bytes of each k-step, of its row in either block
        const char* qa[2];
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const int row = min(row0 + 32 * blk + l32, p.row_end - 1);      // rows past the window repeat the last
            qa[blk] = reinterpret_cast<const char*>(p.q + b * p.qs.b + h * p.qs.h + (int64_t)row * p.qs.s + g * 8);
            if (MASKED && empty[blk]) qa[blk] = reinterpret_cast<const char*>(zero_row + g * 8);
        }

        // LDS -> operands.  K rows (A of S^T): chunk 2 kk + g of row l32 (+ 32).  V^T (A of O^T += V^T P^T),
        // keys in accumulator order: first half rows 16 j + 4 g + r, second half 8 rows further down.
        // The swizzle only touches address bits nothing else sets, so k-step kk (d tile dt) is the first
        // address with kk * 32 (dt * 64) XORed in.
        const int f_row = DH == 128 ? (((l32 & 3) << 2) | ((l32 >> 2) & 3)) : ((((l32 >> 1) & 1) << 2) | ((l32 >> 2) & 3));
        const uint32_t kaddr0 = lds0 + (uint32_t)(l32 * ROWB) + (uint32_t)((g ^ f_row) << 4);
        uint32_t ka[NKK], va[2 * NDT];
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) ka[kk] = kaddr0 ^ (uint32_t)(kk * 32);
        {
            const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
            const int up = DH == 128 ? r : r >> 1;           // the row bits that move a chunk by 64 bytes or more
            const int low = (2 * u + (t >> 1)) ^ g;
            const uint32_t v0 = lds0 + TB + (uint32_t)((4 * g + r) * ROWB + ((4 * up) ^ low) * 16 + (t & 1) * 8);
            const uint32_t v1 = lds0 + TB + (uint32_t)((4 * g + r + 8) * ROWB + ((4 * up) ^ (low ^ 2)) * 16 + (t & 1) * 8);
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) { va[2 * dt] = v0 ^ (uint32_t)(dt * 64); va[2 * dt + 1] = v1 ^ (uint32_t)(dt * 64); }
        }
        const uint32_t me0 = (uint32_t)(my_s[0] - 4 * g), me1 = (uint32_t)(my_s[1] - 4 * g);
        const uint32_t ml0 = (uint32_t)(my_e[0] - my_s[0]), ml1 = (uint32_t)(my_e[1] - my_s[1]);
        // a tile at key kv needs no mask when kv - inner <= inner_n as unsigned numbers
        const bool inner_any = in_hi - in_lo >= BN;
        const int inner = inner_any ? in_lo : BIG;
        const uint32_t inner_n = inner_any ? (uint32_t)(in_hi - BN - in_lo) : 0u;
        uint32_t left = uniform32((uint32_t)(n - 1)), left_k = left, left_v = left, kv = uniform32((uint32_t)kv0);
#define LVX_FWD_WIDE_SCALARS                                                                                       \
    "{s40}"(uniform32(BIAS ? 1.f : p.scale_log2e)), "{s41}"(-INFINITY), "{s42}"(RESCALE_LOG2), "{s48}"(uniform32((uint32_t)BN * krow_b)), \
        "{s49}"(uniform32((uint32_t)BN * vrow_b)), "{s50}"(uniform32(lds_w)), "{s64}"(uniform32((uint32_t)last * krow_b)),   \
        "{s65}"(uniform32((uint32_t)last * vrow_b)), "{s67}"(uniform32(inner)), "{s68}"(uniform32(inner_n)),               \
        "{v224}"(ld_c), "{v225}"(me0), "{v226}"(me1), "{v227}"(ml0), "{v228}"(ml1)
#define LVX_FWD_WIDE_STATE                                                                                         \
    "=&{v229}"(m_i[0]), "=&{v230}"(m_i[1]), "=&{v231}"(l_i[0]), "=&{v232}"(l_i[1]), "+{s[44:45]}"(kp), "+{s[46:47]}"(vp), \
        "+{s51}"(left), "+{s57}"(left_k), "+{s62}"(left_v), "+{s66}"(kv)
#define LVX_FWD_WIDE_OUT_128                                                                                       \
          "=&{v[0:15]}"(acc[0][0]), "=&{v[16:31]}"(acc[0][1]), "=&{v[32:47]}"(acc[0][2]), "=&{v[48:63]}"(acc[0][3]),   \
          "=&{v[64:79]}"(acc[1][0]), "=&{v[80:95]}"(acc[1][1]), "=&{v[96:111]}"(acc[1][2]), "=&{v[112:127]}"(acc[1][3]), \
          "+{v[128:129]}"(qa[0]), "+{v[130:131]}"(qa[1]), "+{v216}"(dok[0]), "+{v217}"(dok[1]), "+{v218}"(dok[2]), "+{v219}"(dok[3]),                              \
          "+{v220}"(dov[0]), "+{v221}"(dov[1]), "+{v222}"(dov[2]), "+{v223}"(dov[3]), LVX_FWD_WIDE_STATE
#define LVX_FWD_WIDE_IN_128                                                                                        \
          "{v200}"(ka[0]), "{v201}"(ka[1]), "{v202}"(ka[2]), "{v203}"(ka[3]), "{v204}"(ka[4]), "{v205}"(ka[5]),    \
          "{v206}"(ka[6]), "{v207}"(ka[7]), "{v208}"(va[0]), "{v209}"(va[1]), "{v210}"(va[2]), "{v211}"(va[3]),    \
          "{v212}"(va[4]), "{v213}"(va[5]), "{v214}"(va[6]), "{v215}"(va[7]), LVX_FWD_WIDE_SCALARS
#define LVX_FWD_WIDE_OUT_64                                                                                        \
          "=&{v[0:15]}"(acc[0][0]), "=&{v[16:31]}"(acc[0][1]), "=&{v[64:79]}"(acc[1][0]), "=&{v[80:95]}"(acc[1][1]),   \
          "+{v[128:129]}"(qa[0]), "+{v[130:131]}"(qa[1]), "+{v216}"(dok[0]), "+{v217}"(dok[1]), "+{v220}"(dov[0]), "+{v221}"(dov[1]), LVX_FWD_WIDE_STATE
#define LVX_FWD_WIDE_IN_64                                                                                         \
          "{v200}"(ka[0]), "{v201}"(ka[1]), "{v202}"(ka[2]), "{v203}"(ka[3]),                                      \
          "{v208}"(va[0]), "{v209}"(va[1]), "{v210}"(va[2]), "{v211}"(va[3]), LVX_FWD_WIDE_SCALARS
        if constexpr (BIAS) {
            // this wave's rows of the bias, from the first tile on.  Loads past the tensor's end give zeros; what they read of rows
            // past the window or of keys past the range is never used.
            const int row = min(row0, p.Lq - 1);
            const float* const base = p.bias + b * p.bias_b + h * p.bias_h + (int64_t)row * p.bias_r + kv0;
            const int64_t bytes = 4 * ((p.Lq - 1 - row) * p.bias_r + (p.Lkv + 3) / 4 * 4 - kv0);
            const uint32_t brow_b = (uint32_t)p.bias_r * 4u;
            const uint64_t at = (uint64_t)(uintptr_t)uniform_ptr(reinterpret_cast<const char*>(base));
            u32x4 srd = {(uint32_t)at, (uint32_t)(at >> 32) & 0xffffu, uniform32((uint32_t)min(bytes, (int64_t)0x7fffffff)), 0x00020000u};
            uint32_t off = (uint32_t)(lane >> 4) * brow_b + (uint32_t)((lane & 15) ^ ((lane >> 4) << 2)) * 16u, left_b = left;
            const uint32_t lds_b = lds0 + 4 * EPB + (uint32_t)wave * BIAS_TILE;
            // chunk 4 m + g (+ 2: the read's offset) of row l32: of block l32 / 4, where its bits 2 and 3 have l32 % 4 XORed in
            u32x4 rd;
#pragma unroll
            for (int m = 0; m < 4; ++m)
                rd[m] = lds_b + (uint32_t)(l32 >> 2) * BIAS_BLOCK + (uint32_t)(l32 & 3) * 256u + (uint32_t)(((4 * m) ^ ((l32 & 3) << 2)) + g) * 16u;
#define LVX_FWD_WIDE_OUT_BIAS "+{v246}"(off), "+{v[248:251]}"(rd), "+{s[72:75]}"(srd), "+{s79}"(left_b)
#define LVX_FWD_WIDE_IN_BIAS "{s76}"(uniform32(4u * brow_b)), "{s77}"(uniform32(lds_b)), "{s78}"(uniform32(p.scale_log2e)), "{s80}"(LOG2E_F)
#define LVX_FWD_WIDE_CLOBBERS_BIAS LVX_FWD_WIDE_CLOBBERS_S, "v245", "v252", "v253", "v254", "v255", "a192", "a193", "a194", "a195"
            if constexpr (DH == 128 && !F16) {
                asm volatile(
#include "lvx_fwd_loop_wide_bf16_128_bias.inc"
                    : LVX_FWD_WIDE_OUT_128, LVX_FWD_WIDE_OUT_BIAS : LVX_FWD_WIDE_IN_128, LVX_FWD_WIDE_IN_BIAS
                    : LVX_FWD_WIDE_CLOBBERS_BIAS, LVX_FWD_WIDE_CLOBBERS_128);
            } else if constexpr (DH == 128) {
                asm volatile(
#include "lvx_fwd_loop_wide_f16_128_bias.inc"
                    : LVX_FWD_WIDE_OUT_128, LVX_FWD_WIDE_OUT_BIAS : LVX_FWD_WIDE_IN_128, LVX_FWD_WIDE_IN_BIAS
                    : LVX_FWD_WIDE_CLOBBERS_BIAS, LVX_FWD_WIDE_CLOBBERS_128);
            } else if constexpr (!F16) {
                asm volatile(
#include "lvx_fwd_loop_wide_bf16_64_bias.inc"
                    : LVX_FWD_WIDE_OUT_64, LVX_FWD_WIDE_OUT_BIAS : LVX_FWD_WIDE_IN_64, LVX_FWD_WIDE_IN_BIAS
                    : LVX_FWD_WIDE_CLOBBERS_BIAS, LVX_FWD_WIDE_CLOBBERS_64);
            } else {
                asm volatile(
#include "lvx_fwd_loop_wide_f16_64_bias.inc"
                    : LVX_FWD_WIDE_OUT_64, LVX_FWD_WIDE_OUT_BIAS : LVX_FWD_WIDE_IN_64, LVX_FWD_WIDE_IN_BIAS
                    : LVX_FWD_WIDE_CLOBBERS_BIAS, LVX_FWD_WIDE_CLOBBERS_64);
            }
            // what a row that sees nothing adds its bias to is not zero times a finite value
#pragma unroll
            for (int blk = 0; blk < 2; ++blk)
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[blk][dt][v] = empty[blk] ? 0.f : acc[blk][dt][v];
        } else if constexpr (DH == 128 && !F16) {
            asm volatile(
#include "lvx_fwd_loop_wide_bf16_128.inc"
                : LVX_FWD_WIDE_OUT_128 : LVX_FWD_WIDE_IN_128 : LVX_FWD_WIDE_CLOBBERS_S, LVX_FWD_WIDE_CLOBBERS_128);
        } else if constexpr (DH == 128) {
            asm volatile(
#include "lvx_fwd_loop_wide_f16_128.inc"
                : LVX_FWD_WIDE_OUT_128 : LVX_FWD_WIDE_IN_128 : LVX_FWD_WIDE_CLOBBERS_S, LVX_FWD_WIDE_CLOBBERS_128);
        } else if constexpr (!F16) {
            asm volatile(
#include "lvx_fwd_loop_wide_bf16_64.inc"
                : LVX_FWD_WIDE_OUT_64 : LVX_FWD_WIDE_IN_64 : LVX_FWD_WIDE_CLOBBERS_S, LVX_FWD_WIDE_CLOBBERS_64);
        } else {
            asm volatile(
#include "lvx_fwd_loop_wide_f16_64.inc"
                : LVX_FWD_WIDE_OUT_64 : LVX_FWD_WIDE_IN_64 : LVX_FWD_WIDE_CLOBBERS_S, LVX_FWD_WIDE_CLOBBERS_64);
        }
    } else {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[blk][dt][v] = 0.f;
    }

    // Epilogue.  A lane holds 4 consecutive values of d of one row per register group; the rows of a wave go through
    // its quarter of the tile buffers and leave as whole rows, 16 bytes per lane.  Rows are 16 bytes longer there
    // than their values, which spreads sixteen of them over the banks and leaves every address a constant away from one
    // register; of rows 16 apart one has the 8-byte halves of its chunks exchanged.  All reads are
    // issued before the first store.  From the last tile to the end 2.1 us; 3.0 with the chunks permuted by XOR, read one by
    // one and stored behind a 64-bit product per row.
    // Parts in fp32 go one block of 32 rows at a time.
    __syncthreads();     // every wave is done with the tiles
    char* const ep = kv_lds + wave * EPB;
    const int64_t o_head = split * p.o_split_stride + b * p.os.b + h * p.os.h + row0 * p.os.s;
    const int rows = p.row_end - row0;                           // of this wave, where fewer than 64
    float l_tot[2], inv[2];
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
        l_tot[blk] = l_i[blk] + __shfl_xor(l_i[blk], 32);       // the two lane halves hold partial sums of the same row
        if (empty[blk]) l_tot[blk] = 0.f;
        inv[blk] = l_tot[blk] > 0.f ? 1.f / l_tot[blk] : 0.f;
    }
    if (p.o_f32) {
        constexpr int CPF = DH / 4, RPS = 64 / CPF;              // chunks of a row of floats, rows per store
        float* const ob = reinterpret_cast<float*>(p.o) + o_head;
        const uint32_t oo = (uint32_t)(lane / CPF) * (uint32_t)p.os.s + (uint32_t)(lane % CPF) * 4u;    // a workspace's stride: DH
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int vg = 0; vg < 4; ++vg) {
                    const f32x4 x = {acc[blk][dt][4 * vg] * inv[blk], acc[blk][dt][4 * vg + 1] * inv[blk],
                                     acc[blk][dt][4 * vg + 2] * inv[blk], acc[blk][dt][4 * vg + 3] * inv[blk]};
                    *reinterpret_cast<f32x4*>(ep + l32 * EP32 + g * 16 + (8 * dt + 2 * vg) * 16) = x;
                }
            wait_lds();
            f32x4 x[32 / RPS];
#pragma unroll
            for (int i = 0; i < 32 / RPS; ++i)
                x[i] = *reinterpret_cast<const f32x4*>(ep + (lane / CPF) * EP32 + (lane % CPF) * 16 + i * (RPS * EP32));
            auto store = [&](bool all) {
#pragma unroll
                for (int i = 0; i < 32 / RPS; ++i) {
                    const int r = 32 * blk + i * RPS;
                    if (all || r + lane / CPF < rows) *reinterpret_cast<f32x4*>(ob + r * p.os.s + oo) = x[i];
                }
            };
            if (rows >= 64) store(true);
            else store(false);
            wait_lds();          // read before the next block takes its place
        }
    } else {
        char* const wr = ep + l32 * EP16 + ((g ^ (l32 >> 4)) << 3);
#pragma unroll
        for (int blk = 0; blk < 2; ++blk)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int vg = 0; vg < 4; ++vg) {
                    u32x2 u;
                    u[0] = E::pack(acc[blk][dt][4 * vg] * inv[blk], acc[blk][dt][4 * vg + 1] * inv[blk]);
                    u[1] = E::pack(acc[blk][dt][4 * vg + 2] * inv[blk], acc[blk][dt][4 * vg + 3] * inv[blk]);
                    *reinterpret_cast<u32x2*>(wr + blk * (32 * EP16) + (4 * dt + vg) * 16) = u;
                }
        wait_lds();          // this wave's rows are its own
        u32x4 x[CPR];
#pragma unroll
        for (int i = 0; i < CPR; ++i) x[i] = *reinterpret_cast<const u32x4*>(ep + (lane / CPR) * EP16 + (lane % CPR) * 16 + i * (RPL * EP16));
        uint16_t* const ob = p.o + o_head + (lane / CPR) * p.os.s + (lane % CPR) * 8;       // a caller's stride: 64 bits
        auto store = [&](bool all) {
#pragma unroll
            for (int i = 0; i < CPR; ++i) {
                const u32x4 y = (i * RPL >> 4) & 1 ? u32x4{x[i][2], x[i][3], x[i][0], x[i][1]} : x[i];
                if (all || i * RPL + lane / CPR < rows) *reinterpret_cast<u32x4*>(ob + i * RPL * p.os.s) = y;
            }
        };
        if (rows >= 64) store(true);
        else store(false);
    }
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
        const int r = 32 * blk + l32;
        if (g == 0 && r < rows) {
            const float lse = l_tot[blk] > 0.f ? m_i[blk] * (BIAS ? LN2_F : p.scale) + __logf(l_tot[blk]) : no_lse(p, l_tot[blk]);
            p.lse[split * p.lse_split_stride + ((int64_t)b * p.Hq + h) * p.lse_bh_stride + row0 + r] = lse;
        }
    }
}

// A launch of the form below whose parts are folded by the work-group that finishes last among those of the same columns (up to four, a
// wave to each; see fold_inside).
//
// They count themselves in at the place of the columns' first four values of O, which nothing else uses before the result
// is written over it: FEW_COUNT above a count of eight bits.  Whatever that memory held, a work-group that does not find FEW_COUNT
// there at its start replaces what it found (and fails to where another has done so), long before anyone counts, so that
// nothing has to be cleared before a launch or kept between two, and a replayed graph counts as the first launch did.
// FEW_COUNT reads as three NaN of bits that no result has.
// Parts and counts go past the L2, of which every XCD has one: stores and loads of agent scope, each step's done (vmcnt) before
// the next begins.
// A launch of its own for the fold takes 4.5 us on the GPU and 3 of the host's time.  In here it is three ways to the memory side one
// behind the other (part, count, parts), 3.4 us: one row x 32 heads x 6404 keys, keys from HBM 11.6 -> 10.1 us a pass, from the cache
// 12.4 -> 9.2; 4 x 1 rows, eight layers with a mask 206 -> 202.5.  (Counting before the sums are formed and waiting for parts that are
// emptied at the start to be filled: 11.8 and 203.5, as the keys then queue behind that.  Loads of one part each and
// reductions through LDS in the fold: 4.2 us.)
constexpr uint64_t FEW_COUNT = 0xffa5ffc37fb95aull;

template <int DH>
struct FewColumns {
    const FwdParams& p;
    const uint32_t ct, b, hk;
    const int rows = p.row_end - p.row_begin, cols = p.G * rows - (int)ct * 32;
    __device__ __forceinline__ uint32_t head(uint32_t col, uint32_t& row) const {
        uint32_t h;
        row = p.by_G.split(ct * 32 + col, h);
        return hk * p.G + h;
    }
    __device__ __forceinline__ uint16_t* o(uint32_t col) const {
        uint32_t row;
        const uint32_t h = head(col, row);
        return p.o + b * p.os.b + (int64_t)h * p.os.h + (int64_t)(p.row_begin + row) * p.os.s;
    }
    __device__ __forceinline__ uint64_t* count() const { return reinterpret_cast<uint64_t*>(o(0)); }
    __device__ __forceinline__ void open(uint64_t found) const {
        if (found >> 8 != FEW_COUNT)
            __hip_atomic_compare_exchange_strong(count(), &found, FEW_COUNT << 8, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ bool last() const {
        return __hip_atomic_fetch_add(count(), 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (FEW_COUNT << 8) + (uint32_t)(p.nsplit - 1);
    }
    // where a column is in a part, and how far apart parts are, in rows
    __device__ __forceinline__ int64_t at(uint32_t col) const {
        uint32_t row;
        const uint32_t h = head(col, row);
        return ((int64_t)b * p.Hq + h) * rows + row;
    }
    __device__ __forceinline__ int64_t all_rows() const { return (int64_t)p.B * p.Hq * rows; }

    // One wave: its column of a part, two values of d to a lane
    __device__ __forceinline__ void store(uint32_t col, uint32_t split, float x0, float x1, float lse) const {
        const int lane = threadIdx.x & 63;
        const int64_t r = split * all_rows() + at(col);
        const uint64_t u = (uint64_t)__float_as_uint(x1) << 32 | __float_as_uint(x0);
        if (lane < DH / 2) __hip_atomic_store(reinterpret_cast<uint64_t*>(p.part + r * DH) + lane, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (lane == 0) __hip_atomic_store(p.l_part + r, lse, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // One wave: a column's parts.  DH / 4 lanes share a part, so that eight loads of the wave have 16 parts of 128 values in
    // flight, and lane k has the weight of part k.
    template <class E>
    __device__ __forceinline__ void fold(uint32_t col) const {
        constexpr int LPP = DH / 4, PPL = 64 / LPP, LOADS = 8;
        const int lane = threadIdx.x & 63, grp = lane / LPP, d = lane % LPP * 4, n = p.nsplit;
        const int64_t all = all_rows(), r = at(col);
        const float* const lp = p.l_part + r + min(lane, n - 1) * all;
        const float* const src = p.part + r * DH + d;
        float l, w = 0.f, m = 0.f, den = 0.f, x[4] = {0.f, 0.f, 0.f, 0.f};
        asm volatile("global_load_dword %0, %1, off sc1" : "=v"(l) : "v"(lp) : "memory");
        int k0 = 0;
        do {
            u32x4 u[LOADS];
#pragma unroll
            for (int j = 0; j < LOADS; ++j)
                asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(u[j]) : "v"(src + min(k0 + j * PPL + grp, n - 1) * (all * DH)) : "memory");
            if (k0 == 0) {
                wait_vmcnt<LOADS>();
                asm volatile("" : "+v"(l));
                if (lane >= n) l = -INFINITY;
                m = wave_max(l);
                w = __expf(l - (m == -INFINITY ? 0.f : m));
                den = wave_sum(w);
            }
            wait_vmcnt<0>();
#pragma unroll
            for (int j = 0; j < LOADS; ++j) asm volatile("" : "+v"(u[j]));
#pragma unroll
            for (int j = 0; j < LOADS; ++j) {
                const int k = k0 + j * PPL + grp;
                float wk = __shfl(w, k & 63);                   // (past the last part: lanes of weight 0)
                if (k >= 64) wk = 0.f;
                // a part of weight 0 may hold anything, one of weight NaN makes the row NaN
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = wk != 0.f ? fmaf(__uint_as_float(u[j][e]), wk, x[e]) : x[e];
            }
        } while ((k0 += LOADS * PPL) < n);
#pragma unroll
        for (int off = LPP; off < 64; off <<= 1)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] += __shfl_xor(x[e], off);
        const float inv = den > 0.f ? 1.f / den : 0.f;
        if (grp == 0) *reinterpret_cast<u32x2*>(o(col) + d) = u32x2{E::pack(x[0] * inv, x[1] * inv), E::pack(x[2] * inv, x[3] * inv)};
        uint32_t row;
        const uint32_t h = head(col, row);
        if (lane == 0) p.lse[((int64_t)b * p.Hq + h) * p.lse_bh_stride + p.row_begin + row] = den > 0.f ? m + __logf(den) : -INFINITY;
    }
};

// Few rows (text being generated, short questions): the work is reading K and V once, 512 bytes per key
// and kv head for a handful of multiplications, so the kernel is built around the loads.
//
// The rows of ALL q heads of a kv head share one 32-column tile (column = row * G + head of the
// group), so K and V are read once per 32 of them.  A work-group is 4 waves on one key range; each wave
// takes every fourth 32-key piece, loads it straight into a ring of two pieces of its own in LDS and
// works on it alone - no barrier until the four partial results are folded at the end.  Both pieces
// are requested before anything else happens: 128 KiB in flight per CU, and with ranges of 256 keys
// or less every byte the work-group will read.  Bound by HBM where there is enough to read: 4 rows x 32
// heads x 76848 keys (315 MB) take 61 us, 5.2 TB/s, the rate of a large copy, against 75 us in the
// wide form; one row x 6404 keys (26 MB) 10.1 us with the fold of the parts inside against 17.4 in two launches, most of
// it latency (9.1 us in the kernel, 6.1 without the fold; 6.7 with the arguments fetched line by line and integer divisions for where it is).
//   S^T[32 keys, 32 cols] = K (A, 16-byte LDS reads) x Q^T (B, registers)
//   O^T[d, 32 cols]      += V^T (A, transposing LDS reads) x P^T (B, straight from S^T)
// LDS rows are 2 DH bytes (128 below head dimension 64, the lanes past the head dimension repeat a
// chunk of the row), chunks permuted as in fwd_wide_kernel.
// INSIDE (fwd_fewest_kernel): the launch folds its own parts (a test at run time costs every other launch 0.2 us: four rounds of 140 rows x 3 heads of 32 35.6
// us a pass without it, 36.3 with).
template <int DH, bool MASKED, bool F16, bool INSIDE>
__device__ __forceinline__ void fwd_few(const FwdParams& p) {
    using E = Elt<F16>;
    constexpr int LW = DH >= 64 ? DH : 64;                          // elements per LDS row
    constexpr int NKK = DH / 16, NDT = DH >= 32 ? DH / 32 : 1;
    constexpr int ROWB = 2 * LW, CPR = LW / 8, RPL = 64 / CPR;      // bytes and chunks per row, rows per load
    constexpr int PB = 32 * ROWB, NLD = PB / 1024;                  // bytes and loads of a K (or V) piece
    constexpr int EPS = 32 * NDT + 4;                               // row stride (floats) of the fold tile
    constexpr int RING = 4 * 2 * 2 * PB, FOLD = 4 * 32 * EPS * 4;
    __shared__ __attribute__((aligned(1024))) char lds[RING > FOLD ? RING : FOLD];
    __shared__ float ml[4][2][32];                                  // per wave and column: reference maximum, row sum

    fetch_kernargs<sizeof(FwdParams)>();
    const int wid = xcd_remap(blockIdx.x, p.total_wg);
    if (wid >= p.total_wg) return;
    uint32_t ct, split, b;                         // column tile, key range, sample
    const uint32_t t1 = p.by_row_tiles.split(wid, ct), t2 = p.by_splits.split(t1, split), hk = p.by_B.split(t2, b);

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int n_cols = p.G * (p.row_end - p.row_begin);
    const int col = min((int)ct * 32 + l32, n_cols - 1);            // columns past the last repeat it and are not stored
    uint32_t head;
    const int row = p.row_begin + p.by_G.split(col, head), h = hk * p.G + head;

    const FewColumns<DH> columns{p, ct, b, hk};     // (INSIDE)
    uint64_t word = 0;
    if constexpr (INSIDE) asm volatile("global_load_dwordx2 %0, %1, off sc1" : "=v"(word) : "v"(columns.count()) : "memory");

    u32x4 q[NKK];
    {
        const char* qp = reinterpret_cast<const char*>(p.q + b * p.qs.b + h * p.qs.h + (int64_t)row * p.qs.s + g * 8);
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk)
            asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "=v"(q[kk]) : "v"(qp), "n"(32 * kk));
    }

    int kv_len = p.Lkv;
    if (p.kv_len) kv_len = min(p.kv_len[b], p.Lkv);
    const int kv_lo = split * p.split_len;
    const int kv_hi = min(kv_len, kv_lo + p.split_len);
    int my_s = kv_lo, my_e = kv_hi, lo = kv_lo, hi = kv_hi, in_lo = kv_lo, in_hi = kv_hi;
    bool empty = kv_hi <= kv_lo;
    if (MASKED) {
        my_s = max(kv_lo, p.kv_start[(int64_t)b * p.Lq + row]);
        my_e = min(kv_hi, p.kv_end[(int64_t)b * p.Lq + row]);
        empty = my_e <= my_s;
        // a row that sees nothing is let see everything, with a Q of zeros, and stored as zeros (see fwd_wide_kernel)
        lo = empty ? BIG : my_s; hi = empty ? 0 : my_e;
        in_lo = empty ? 0 : my_s; in_hi = empty ? BIG : my_e;
        if (empty) { my_s = 0; my_e = BIG; }
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) {      // the two halves of a wave hold the same columns
            lo = min(lo, __shfl_xor(lo, off));
            hi = max(hi, __shfl_xor(hi, off));
            in_lo = max(in_lo, __shfl_xor(in_lo, off));
            in_hi = min(in_hi, __shfl_xor(in_hi, off));
        }
        lo = uniform32(lo); hi = uniform32(hi); in_lo = uniform32(in_lo); in_hi = uniform32(in_hi);
    }
    const int base = lo / 32 * 32;
    const int n_piece = hi > lo ? (hi - base + 31) / 32 : 0;
    const int n = n_piece > wave ? (n_piece - wave + 3) / 4 : 0;    // pieces of this wave

    const char* const kbase = reinterpret_cast<const char*>(p.k + b * p.ks.b + hk * p.ks.h);
    const char* const vbase = reinterpret_cast<const char*>(p.v + b * p.vs.b + hk * p.vs.h);
    const uint32_t krow_b = (uint32_t)p.ks.s * 2u, vrow_b = (uint32_t)p.vs.s * 2u;
    const uint32_t ring = (uint32_t)(uintptr_t)&lds[0] + (uint32_t)wave * (4 * PB);
    const int ld_r = lane / CPR;
    auto issue = [&](int i) {       // this wave's piece i into ring slot i & 1; rows past the last key repeat it
        const int kv0 = base + 32 * (wave + 4 * i);
        const char* kb = uniform_ptr(kbase + (int64_t)kv0 * krow_b);
        const char* vb = uniform_ptr(vbase + (int64_t)kv0 * vrow_b);
        const uint32_t slot = uniform32(ring + (uint32_t)(i & 1) * (2 * PB));
        const int last = hi - 1 - kv0;
#pragma unroll
        for (int j = 0; j < NLD; ++j) {
            const uint32_t r = (uint32_t)min(RPL * j + ld_r, last);
            const int f = LW == 128 ? ((lane >> 4) << 2) | (j & 3) : (((lane >> 4) & 1) << 2) | ((2 * j + (lane >> 5)) & 3);
            const uint32_t c = (uint32_t)(((lane % CPR) ^ f) & (DH / 8 - 1)) * 16u;
            dma16(kb, r * krow_b + c, slot + j * 1024);
            dma16(vb, r * vrow_b + c, slot + PB + j * 1024);
        }
    };
    if (n > 0) issue(0);
    if (n > 1) issue(1);

    // LDS -> operands, as in fwd_wide_kernel
    const int f_row = LW == 128 ? (((l32 & 3) << 2) | ((l32 >> 2) & 3)) : ((((l32 >> 1) & 1) << 2) | ((l32 >> 2) & 3));
    const uint32_t k_rd = (uint32_t)(l32 * ROWB) + (uint32_t)((g ^ f_row) << 4);
    uint32_t v_rd[2];
    {
        const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
        const int up = LW == 128 ? r : r >> 1, low = (2 * u + (t >> 1)) ^ g;
        v_rd[0] = PB + (uint32_t)((4 * g + r) * ROWB + ((4 * up) ^ low) * 16 + (t & 1) * 8);
        v_rd[1] = PB + (uint32_t)((4 * g + r + 8) * ROWB + ((4 * up) ^ (low ^ 2)) * 16 + (t & 1) * 8);
    }

    f32x16 acc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[dt][v] = 0.f;
    float m_i = -INFINITY, l_i = 0.f;
    const float cc = p.scale_log2e;

    // Q was requested first: it is here when at most two pieces' loads are outstanding (with fewer of them, when
    // nothing is).  The compiler takes q for loaded from its request on, so nothing must make it touch those
    // registers before this wait, which is one statement that every path comes by; the tests follow
    // the paths of the built code from the request to here.
    asm volatile("s_cmp_gt_i32 %0, 1\n\ts_cbranch_scc1 LVX_FEW_TWO_%=\n\ts_waitcnt vmcnt(0)\nLVX_FEW_TWO_%=:\n\ts_waitcnt vmcnt(%1)"
                 ::"s"(uniform32(n)), "n"(4 * NLD) : "memory", "scc");
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
        asm volatile("" : "+v"(q[kk]));
        if (MASKED && empty) q[kk] = u32x4{0u, 0u, 0u, 0u};
    }
    if constexpr (INSIDE) {
        asm volatile("" : "+v"(word));      // requested before Q
        if (tid == 0) columns.open(word);
    }

    for (int i = 0; i < n; ++i) {
        const int kv0 = base + 32 * (wave + 4 * i);
        const char* const pc = lds + wave * (4 * PB) + (i & 1) * (2 * PB);
        if (i + 1 < n) wait_vmcnt<2 * NLD>();
        else wait_vmcnt<0>();
        f32x16 s;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
            const bf16x8 ka = *reinterpret_cast<const bf16x8*>(pc + (k_rd ^ (uint32_t)(kk * 32)));
            s = E::mfma(ka, as_bf16x8(q[kk]), s);
        }
        u32x2 va[NDT][2][2];        // requested now, they land during the softmax
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    va[dt][j][e] = lds_read_tr16(reinterpret_cast<const uint16_t*>(pc + (v_rd[e] ^ (uint32_t)(dt * 64)) + j * 16 * ROWB));
        if (kv0 < in_lo || kv0 + 32 > in_hi) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int kv = kv0 + acc_row(v, g);
                if (kv < my_s || kv >= my_e) s[v] = -INFINITY;
            }
        }
        mfma_settle(s);
        float mx = max3(s[0], s[1], s[2]);
#pragma unroll
        for (int v = 3; v < 15; v += 2) mx = max3(mx, s[v], s[v + 1]);
        mx = fmaxf(mx, s[15]);
        {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = max3(__uint_as_float(sw[0]), __uint_as_float(sw[1]), m_i);
        }
        // lazy rescale, as in fwd_kernel
        const float mcand = mx * cc, m_ic = m_i * cc;
        const bool move = (mx != -INFINITY) && !(mcand - m_ic <= RESCALE_LOG2);
        const float alpha = move ? __builtin_amdgcn_exp2f(m_ic - mcand) : 1.f;
        if (move) m_i = mx;
        const float mc = (m_i == -INFINITY) ? 0.f : m_i * cc;
        bf16x8 pb[2];
        float rs = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            u32x4 u;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a0 = __builtin_amdgcn_exp2f(fmaf(s[8 * j + 2 * e], cc, -mc)), a1 = __builtin_amdgcn_exp2f(fmaf(s[8 * j + 2 * e + 1], cc, -mc));
                rs += a0 + a1;
                u[e] = E::pack(a0, a1);
            }
            pb[j] = as_bf16x8(u);
        }
        l_i = l_i * alpha + rs;
        if (i > 0 && __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[dt][v] *= alpha;
        }
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const u32x4 a = {va[dt][j][0][0], va[dt][j][0][1], va[dt][j][1][0], va[dt][j][1][1]};
                acc[dt] = E::mfma(as_bf16x8(a), pb[j], acc[dt]);
            }
        if (i + 2 < n) {
            wait_lds();             // this slot has been read
            issue(i + 2);
        }
    }

    // Fold the four waves: every wave leaves its O^T as rows [col][d] in fp32 with its reference and sum;
    // 8 lanes then share a column.
    __syncthreads();                // the ring is free
    float* const ep = reinterpret_cast<float*>(lds) + wave * (32 * EPS);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int vg = 0; vg < 4; ++vg) {
            const f32x4 x = {acc[dt][4 * vg], acc[dt][4 * vg + 1], acc[dt][4 * vg + 2], acc[dt][4 * vg + 3]};
            *reinterpret_cast<f32x4*>(ep + l32 * EPS + dt * 32 + 8 * vg + 4 * g) = x;
        }
    const float l_tot = l_i + __shfl_xor(l_i, 32);
    if (g == 0) {
        ml[wave][0][l32] = m_i;
        ml[wave][1][l32] = empty ? 0.f : l_tot;
    }
    __syncthreads();
    if constexpr (INSIDE) {         // the columns are four at most
        if (wave < columns.cols) {
            float M = -INFINITY, den = 0.f, x0 = 0.f, x1 = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) M = fmaxf(M, ml[k][0][wave]);
            const float* const src = reinterpret_cast<const float*>(lds) + wave * EPS + 2 * min(lane, DH / 2 - 1);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float w = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((ml[k][0][wave] - M) * cc);
                den = fmaf(w, ml[k][1][wave], den);
                x0 = fmaf(w, src[k * (32 * EPS)], x0);
                x1 = fmaf(w, src[k * (32 * EPS) + 1], x1);
            }
            const float inv = den > 0.f ? 1.f / den : 0.f;
            columns.store(wave, split, x0 * inv, x1 * inv, den > 0.f ? M * p.scale + __logf(den) : no_lse(p, den));
            wait_vmcnt<0>();        // it is where the last work-group will read it
        }
        __syncthreads();
        __shared__ int last;
        if (tid == 0) last = columns.last();
        __syncthreads();
        if (last && wave < columns.cols) columns.template fold<E>(wave);
        return;
    }
    constexpr int TPC = 8, DPT = DH / TPC;          // threads per column, values of d per thread
    const int oc = tid / TPC, part = tid % TPC;
    if ((int)ct * 32 + oc >= n_cols) return;
    const int orow = p.row_begin + p.by_G.split(ct * 32 + oc, head), oh = hk * p.G + head;
    float M = -INFINITY, w[4], den = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) M = fmaxf(M, ml[k][0][oc]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        w[k] = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((ml[k][0][oc] - M) * cc);
        den = fmaf(w[k], ml[k][1][oc], den);
    }
    const float inv = den > 0.f ? 1.f / den : 0.f;
    const int64_t at = split * p.o_split_stride + b * p.os.b + oh * p.os.h + (int64_t)orow * p.os.s + part * DPT;
    uint16_t* const op = p.o + at;
    float* const op32 = reinterpret_cast<float*>(p.o) + at;
    const float* const src = reinterpret_cast<const float*>(lds) + oc * EPS + part * DPT;
    uint32_t out[DPT / 2];
    float out32[DPT];
#pragma unroll
    for (int d = 0; d < DPT; d += 2) {
        float x0 = 0.f, x1 = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x0 = fmaf(w[k], src[k * (32 * EPS) + d], x0);
            x1 = fmaf(w[k], src[k * (32 * EPS) + d + 1], x1);
        }
        out32[d] = x0 * inv;
        out32[d + 1] = x1 * inv;
        out[d / 2] = E::pack(out32[d], out32[d + 1]);
    }
    if (p.o_f32) {
#pragma unroll
        for (int d = 0; d < DPT; d += 2) *reinterpret_cast<float2*>(op32 + d) = float2{out32[d], out32[d + 1]};
    } else if constexpr (DPT >= 8) {
#pragma unroll
        for (int d = 0; d < DPT / 8; ++d)
            *reinterpret_cast<u32x4*>(op + 8 * d) = u32x4{out[4 * d], out[4 * d + 1], out[4 * d + 2], out[4 * d + 3]};
    } else {
#pragma unroll
        for (int d = 0; d < DPT / 2; ++d) *reinterpret_cast<uint32_t*>(op + 2 * d) = out[d];
    }
    if (part == 0)
        p.lse[split * p.lse_split_stride + ((int64_t)b * p.Hq + oh) * p.lse_bh_stride + orow] =
            den > 0.f ? M * p.scale + __logf(den) : no_lse(p, den);
}
template <int DH, bool MASKED, bool F16>
__global__ __launch_bounds__(256, 1) void fwd_few_kernel(const FwdParams p) { fwd_few<DH, MASKED, F16, false>(p); }
template <int DH, bool MASKED, bool F16>
__global__ __launch_bounds__(256, 1) void fwd_fewest_kernel(const FwdParams p) { fwd_few<DH, MASKED, F16, true>(p); }

}  // namespace

namespace {
template <int DH, bool F16>
hipError_t launch_fwd_t(const FwdParams& p, bool masked, hipStream_t st, const FwdFold* fold = nullptr) {
    const int grid = ((p.total_wg + 7) / 8) * 8;
    if (p.form == FWD_FEW) {
        if (p.part) {
            if (masked) return launch1((fwd_fewest_kernel<DH, true, F16>), dim3(grid), dim3(256), st, p);
            return launch1((fwd_fewest_kernel<DH, false, F16>), dim3(grid), dim3(256), st, p);
        }
        if (masked) return launch1((fwd_few_kernel<DH, true, F16>), dim3(grid), dim3(256), st, p);
        return launch1((fwd_few_kernel<DH, false, F16>), dim3(grid), dim3(256), st, p);
    }
    if constexpr (DH >= 64) {
        if (p.form == FWD_WIDE) {
            if (p.bias) return launch1((fwd_wide_kernel<DH, true, F16, false, true>), dim3(grid), dim3(256), st, p);
            if (fold) {
                const FwdFoldParams both{p, *fold};
                if (masked) return launch1((fwd_wide_kernel<DH, true, F16, true>), dim3(grid), dim3(256), st, both);
                return launch1((fwd_wide_kernel<DH, false, F16, true>), dim3(grid), dim3(256), st, both);
            }
            if (masked) return launch1((fwd_wide_kernel<DH, true, F16, false>), dim3(grid), dim3(256), st, p);
            return launch1((fwd_wide_kernel<DH, false, F16, false>), dim3(grid), dim3(256), st, p);
        }
        if (!p.bias) return hipErrorInvalidValue;      // fwd_form never asks for it
    }
    if (p.bias) {
        if (masked) return launch1((fwd_kernel<DH, true, true, F16>), dim3(grid), dim3(256), st, p);
        return launch1((fwd_kernel<DH, false, true, F16>), dim3(grid), dim3(256), st, p);
    }
    if constexpr (DH < 64) {
        if (masked) return launch1((fwd_kernel<DH, true, false, F16>), dim3(grid), dim3(256), st, p);
        return launch1((fwd_kernel<DH, false, false, F16>), dim3(grid), dim3(256), st, p);
    }
    return hipErrorInvalidValue;
}
}  // namespace

hipError_t launch_fwd(const FwdParams& params, bool masked, hipStream_t st, const FwdFold* before) {
    FwdParams p = params;
    p.by_row_tiles = divisor(p.n_row_tiles);
    p.by_splits = divisor(p.nsplit);
    p.by_B = divisor(p.B);
    p.by_G = divisor(p.G);
    p.by_head_groups = divisor(p.G / p.HG);
    if (before) {
        FwdFold fold = *before;
        const int64_t rows = (int64_t)p.B * p.Hq * fold.rows;
        if (p.form != FWD_WIDE || !fold_rides(fold.nparts, rows, p.D / 8, p.total_wg, cu_count())) return hipErrorInvalidValue;
        fold.chains = fold_chains(fold.nparts, rows);
        fold.per_wg = (uint32_t)fold_per_wg(rows, p.D / 8, p.total_wg);
        fold.by_rows = divisor(fold.rows);
        if (p.D == 128) return p.f16 ? launch_fwd_t<128, true>(p, masked, st, &fold) : launch_fwd_t<128, false>(p, masked, st, &fold);
        return p.f16 ? launch_fwd_t<64, true>(p, masked, st, &fold) : launch_fwd_t<64, false>(p, masked, st, &fold);
    }
    switch (p.D) {
        case 16: return p.f16 ? launch_fwd_t<16, true>(p, masked, st) : launch_fwd_t<16, false>(p, masked, st);
        case 32: return p.f16 ? launch_fwd_t<32, true>(p, masked, st) : launch_fwd_t<32, false>(p, masked, st);
        case 64: return p.f16 ? launch_fwd_t<64, true>(p, masked, st) : launch_fwd_t<64, false>(p, masked, st);
        case 128: return p.f16 ? launch_fwd_t<128, true>(p, masked, st) : launch_fwd_t<128, false>(p, masked, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace lvx

// dQ = (scale dS) K of the attention backward, from the dS^T workspace that bwd_kernel leaves: per (sample, q head) a
// product [rows x tokens] [tokens x head dimension] whose left operand is read from memory exactly once.
#include <cstddef>

#include "lvx_common.hpp"
#include "lvx_fold.hpp"
#include "lvx_dq_rule.hpp"
#include "lvx_kernels.hpp"

#include <type_traits>

namespace lvx {

namespace {

// A work-group takes 256 rows of one head, each of its four waves two 32-row tiles of dS^T and all of the head dimension,
// alone on its SIMD.  bwd_kernel leaves a tile as [token / 8][row][8 tokens], which is this product's operand: a load of a
// wave is 1 KiB in a row and goes straight into the registers the MFMA reads, past the LDS and past every other wave.  K is
// shared, in LDS rows of LW elements whose 64-byte groups are permuted by the token so that the four rows of a transposing
// read lie in different banks.  Stages of 32 tokens (16 KiB of dS^T; 8 of K, 4 with heads up to 64), NS of them in
// registers and LDS, one barrier a stage, behind which the next one is requested.
//   dQ^T[d, row] += K^T (A, transposing LDS reads) x dS^T (B, from memory)
// Bound by reading dS^T: 4096 rows x 32 heads x 6404 tokens (1.7 GB) 280 us, 6.0 TB/s; heads of 64, 2048 rows (0.84 GB) 130 us.
// The eight-wave form that this replaces (dS^T through LDS in [token][row] tiles, two sets of waves in turn, two barriers a
// stage of 32) took 311 and 159, rounds of 256 rows 27.4 where this takes 24.8, 2 x 3000 rows with image intervals 237, 199
// now - and more power, which the chip takes from the kernels beside it: with eight waves that each took
// 32 rows from LDS, as fast as this one, sixteen rounds forward and backward were slower than before (2862 -> 2879 us; 2805 ->
// 2786 with this one).  With three, four or five stages in the ring instead, or one work-group per CU instead of the
// two that the registers leave room for, within 0.3 % of each other.
// RANGED: a row tile counts inside its own range of tokens only (tile_range); outside, its loads are sent out of
// the descriptor's range: they give zeros and read nothing.
template <int DH, bool F16, bool STREAM, bool RANGED>
__global__ __launch_bounds__(256, 1) void dq_kernel(const DqParams p) {
    using E = Elt<F16>;
    static_assert(DH == 16 || DH == 32 || DH == 64 || DH == 128, "head dimension");
    constexpr int LW = DH >= 64 ? DH : 64, NDT = DH >= 32 ? DH / 32 : 1;
    constexpr int BK = 32, NS = LW == 128 ? 5 : 6;
    constexpr int ROWB = 2 * LW, CPR = LW / 8, RPL = 64 / CPR;      // bytes, chunks of a K row, rows per load
    constexpr int STAGE = BK * ROWB, NKL = STAGE / 4096, NL = 4 + NKL;          // K's bytes and loads, all loads of a wave per stage
    constexpr int EP = 2 * DH + 16;                                 // row stride of the tile that dQ leaves through
    constexpr int RING = NS * STAGE, OUT = 4 * 32 * EP;
    __shared__ __attribute__((aligned(1024))) char lds[RING > OUT ? RING : OUT];

    fetch_kernargs<offsetof(DqParams, cast)>();
    if ((int)blockIdx.x < p.cast_wg) { cast_slices<F16>(p.cast, blockIdx.x); return; }
    const int wid = p.order ? (int)blockIdx.x - p.cast_wg : xcd_remap(blockIdx.x - p.cast_wg, p.total_wg);
    if (wid >= p.total_wg) return;
    uint32_t split, tm, b, h;
    const uint32_t t1 = p.by_splits.split(wid, split);
    if (p.order) {
        // groups of row tiles ranked by the length of their contraction: the ids walk the ranking, heads fastest, so that
        // the hardware's in-order hand-out starts the longest first, on every XCD alike
        b = p.by_tiles_m.split((uint32_t)p.order[p.by_Hq.split(t1, h)], tm);
    } else {
        h = p.by_B.split(p.by_tiles_m.split(t1, tm), b);       // samples fastest: every XCD gets work of all of them
    }
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int tile0 = (int)tm * 8 + 2 * wave;           // this wave's first row tile

    int k_lo = 0, k_hi = p.Lkv;
    if (p.kv_len) k_hi = min(k_hi, p.kv_len[b]);
    if (p.k_splits > 1) { k_lo = (int)split * p.split_len; k_hi = min(k_hi, k_lo + p.split_len); }
    uint32_t a_lo[2], a_len[2];                         // tokens at which this wave's tiles count
#pragma unroll
    for (int i = 0; i < 2; ++i) { a_lo[i] = 0; a_len[i] = tile0 + i < p.row_tiles ? 0x7fffffffu : 0u; }
    if (RANGED) {
        const int32_t* range = p.tile_range + (int64_t)b * p.row_tiles * 2;
        const int t = min((int)tm * 8 + (lane & 7), p.row_tiles - 1);
        int lo = range[2 * t], hi = range[2 * t + 1];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            a_lo[i] = (uint32_t)__builtin_amdgcn_readlane(lo, 2 * wave + i);
            if (a_len[i]) a_len[i] = (uint32_t)__builtin_amdgcn_readlane(hi, 2 * wave + i) - a_lo[i];
        }
        if (hi == 0) lo = 0x7fffffff;
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) {
            lo = min(lo, __shfl_xor(lo, off));
            hi = max(hi, __shfl_xor(hi, off));
        }
        k_hi = min(k_hi, uniform32(hi));
        k_lo = max(k_lo, min(uniform32(lo), uniform32(hi)));
    }
    k_hi = uniform32(k_hi);
    k_lo = uniform32(k_lo);
    const int steps = k_hi > k_lo ? (k_hi - k_lo + BK - 1) / BK : 0;

    // dS^T -> registers: stage by stage [k-step][tile].  Ranges of tokens begin with a block of 128.
    u32x4 ds[NS][2][2];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) ds[s][i >> 1][i & 1] = u32x4{0u, 0u, 0u, 0u};
    const char* a_ptr = uniform_ptr(reinterpret_cast<const char*>(p.ds + ((int64_t)b * p.Hq + h) * p.ds_bh) +
                                    ((int64_t)(k_lo >> 7) * p.row_tiles + min(tile0, p.row_tiles - 1)) * 8192);
    const int64_t a_jump = (int64_t)(p.row_tiles - 1) * 8192;       // behind a tile's last stage
    // K -> LDS
    const uint32_t krow_b = (uint32_t)p.ks.s * 2u;
    const char* b_ptr = uniform_ptr(reinterpret_cast<const char*>(p.k + b * p.ks.b + p.by_G.quotient(h) * p.ks.h) + (int64_t)k_lo * krow_b);
    const uint32_t lds_w = (uint32_t)(uintptr_t)lds + (uint32_t)wave * 1024u;
    const int b_row = RPL * wave + lane / CPR;                      // and 4 RPL further in the second load
    const uint32_t b_chunk = (uint32_t)(((lane % CPR) ^ (LW == 128 ? (lane >> 4) << 2 : ((lane >> 4) & 1) << 2)) & (DH / 8 - 1)) * 16u;
    const uint32_t b_off = (uint32_t)b_row * krow_b + b_chunk;
    int k_next = k_lo;                                              // first token of the stage to request
    auto issue = [&](u32x4 (&to)[2][2], int slot) __attribute__((always_inline)) {
        const uint64_t a = (uint64_t)(uintptr_t)a_ptr;
        const u32x4 srd = {(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, 16384u, 0x00020000u};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t off = (uint32_t)lane * 16u + ((uint32_t)k_next - a_lo[i] < a_len[i] ? 8192u * i : 0x80000000u);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                if (STREAM) asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen offset:%3 nt" : "+v"(to[kk][i]) : "v"(off), "s"(srd), "n"(1024 * kk));
                else asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen offset:%3" : "+v"(to[kk][i]) : "v"(off), "s"(srd), "n"(1024 * kk));
        }
        const int last = k_hi - 1 - k_next;             // rows of K past the last one repeat it: dS^T is zero there
#pragma unroll
        for (int j = 0; j < NKL; ++j) {
            uint32_t off = b_off + (uint32_t)(4 * RPL * j) * krow_b;
            if (last < BK - 1) off = (uint32_t)min(b_row + 4 * RPL * j, last) * krow_b + b_chunk;
            dma16(b_ptr, off, lds_w + slot * STAGE + j * 4096);
        }
        k_next += BK;
        a_ptr += 2048;
        if ((k_next & 127) == 0) a_ptr += a_jump;
        b_ptr += (int64_t)BK * krow_b;
    };

    // K^T from LDS, tokens in natural order: the second half of a k-step's eight is four rows further down
    const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
    uint32_t b_rd[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
        b_rd[dt] = (uint32_t)((8 * g + r) * ROWB + 64 * (dt ^ (LW == 128 ? r : r >> 1)) + (2 * u + (t >> 1)) * 16 + (t & 1) * 8);

    f32x16 acc[2][NDT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][dt][v] = 0.f;

#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < steps) issue(ds[s], s);
    int k_at = k_lo;
    for (int s0 = 0; s0 < steps; s0 += NS) {
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int s = s0 + i;
            if (s >= steps) break;
            // one statement that every path comes by: the registers are in flight until here
            asm volatile("s_cmp_ge_i32 %0, %1\n\ts_cbranch_scc1 LVX_DQ_MORE_%=\n\ts_waitcnt vmcnt(0)\nLVX_DQ_MORE_%=:\n\ts_waitcnt vmcnt(%2)"
                         ::"s"(uniform32(steps - s)), "n"(NS - 1), "n"((NS - 2) * NL) : "memory", "scc");
#pragma unroll
            for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(ds[i][j >> 1][j & 1]));
            lds_barrier();      // every wave's part of K has landed, and the stage before has been read
            if (s + NS - 1 < steps) issue(ds[(i + NS - 1) % NS], (i + NS - 1) % NS);
            if (k_at + BK > k_hi) {         // the last stage: tokens past the end count as zeros
#pragma unroll
                for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const int left = k_hi - (k_at + 16 * kk + 8 * g + 2 * w);
                        const uint32_t keep = left >= 2 ? 0xffffffffu : left == 1 ? 0xffffu : 0u;
                        ds[i][kk][0][w] &= keep;
                        ds[i][kk][1][w] &= keep;
                    }
            }
            const char* const st = lds + i * STAGE;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    const bf16x8 kt = lds_operand_tr(reinterpret_cast<const uint16_t*>(st + b_rd[dt] + kk * 16 * ROWB), 4 * LW);
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[j][dt] = E::mfma(kt, as_bf16x8(ds[i][kk][j]), acc[j][dt]);
                }
            k_at += BK;
        }
    }

    // dQ^T: rows = d, columns = text rows
    if (p.k_splits > 1) {       // partial tiles, fp32, in this split's slice [B * Hq][DH][rows]: 128 bytes a store
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = (tile0 + j) * 32 + l32;
            if (row >= p.rows) continue;
            float* const c = p.part + split * p.part_split + ((int64_t)b * p.Hq + h) * DH * p.rows + row;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (dt * 32 + 8 * (v >> 2) < DH) c[(int64_t)(dt * 32 + acc_row(v, g)) * p.rows] = acc[j][dt][v];
        }
        return;
    }
    // The tiles turn through this wave's part of the LDS and leave as whole rows (see fwd_wide_kernel's epilogue).
    __syncthreads();            // every wave is done with K
    constexpr int CPO = DH / 8, RPS = 64 / CPO;                     // chunks of a row of dQ, rows per store
    char* const ep = lds + wave * (32 * EP);
    uint16_t* const out = p.dq + b * p.dqs.b + h * p.dqs.h + (lane % CPO) * 8;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row0 = (tile0 + j) * 32;
        if (row0 >= p.rows) return;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int vg = 0; vg < 4; ++vg) {
                if (dt * 32 + 8 * vg >= DH) continue;
                const u32x2 x = {E::pack(acc[j][dt][4 * vg], acc[j][dt][4 * vg + 1]), E::pack(acc[j][dt][4 * vg + 2], acc[j][dt][4 * vg + 3])};
                *reinterpret_cast<u32x2*>(ep + l32 * EP + (4 * dt + vg) * 16 + ((g ^ (l32 >> 4)) << 3)) = x;
            }
        wait_lds();
#pragma unroll
        for (int i = 0; i < 32 / RPS; ++i) {
            const int row = i * RPS + lane / CPO;
            u32x4 x = *reinterpret_cast<const u32x4*>(ep + row * EP + (lane % CPO) * 16);
            if (row >> 4) x = u32x4{x[2], x[3], x[0], x[1]};
            // (a streaming store: nobody on this CU reads the tile again)
            if (row0 + row < p.rows) __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(out + (int64_t)(row0 + row) * p.dqs.s));
        }
        wait_lds();             // read before the next tile takes its place
    }
}

// The same for windows of few rows: a work-group takes 64 rows (two tiles) and its four waves share the TOKENS, every
// fourth stage of 32 each, with K in rings of their own - no barrier until the four sums are added in LDS at the end.  Four times
// as many work-groups as the form above at four times the reads of K (from the L2), so that it is for launches where that one's
// are fewer than half the CUs: those had to cut the contraction into up to eight ranges, whose fp32 slices are written by all
// of them at once when they end and summed by another launch.  us, with the sum: 1024 rows x 16 heads x 4096 tokens 33.0 + 7.7 (four
// ranges) -> 27.7 (one), 256 rows x 32 heads x 6404 tokens 24.8 + 7.1 (eight) -> 24.1 + 5.1 (two): bound by K's way from the
// L2, twice the bytes of dS^T.
template <int DH, bool F16, bool STREAM, bool RANGED>
__global__ __launch_bounds__(256, 1) void dq_few_kernel(const DqParams p) {
    using E = Elt<F16>;
    constexpr int LW = DH >= 64 ? DH : 64, NDT = DH >= 32 ? DH / 32 : 1;
    constexpr int BK = 32, NS = 4;
    constexpr int ROWB = 2 * LW, CPR = LW / 8, RPL = 64 / CPR;      // bytes, chunks of a K row, rows per load
    constexpr int STAGE = BK * ROWB, NKL = STAGE / 1024, NL = 4 + NKL;          // K's bytes and loads, all loads of a wave per stage
    constexpr int CW = DH / 16, EP = CW * 16 + 16;                  // 8-value chunks of a row that a wave sums, their row stride
    constexpr int RING = 4 * NS * STAGE, SUMS = 4 * 2 * 2 * CW * 1024;
    __shared__ __attribute__((aligned(1024))) char lds[RING > SUMS ? RING : SUMS];
    static_assert(4 * 32 * EP <= RING);

    fetch_kernargs<offsetof(DqParams, cast)>();
    if ((int)blockIdx.x < p.cast_wg) { cast_slices<F16>(p.cast, blockIdx.x); return; }
    const int wid = xcd_remap(blockIdx.x - p.cast_wg, p.total_wg);
    if (wid >= p.total_wg) return;
    uint32_t split, tm, b;
    const uint32_t t1 = p.by_splits.split(wid, split);
    const uint32_t h = p.by_B.split(p.by_tiles_m.split(t1, tm), b);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int tile0 = (int)tm * 2;

    int k_lo = 0, k_hi = p.Lkv;
    if (p.kv_len) k_hi = min(k_hi, p.kv_len[b]);
    if (p.k_splits > 1) { k_lo = (int)split * p.split_len; k_hi = min(k_hi, k_lo + p.split_len); }
    uint32_t a_lo[2], a_len[2];                         // tokens at which the tiles count
#pragma unroll
    for (int i = 0; i < 2; ++i) { a_lo[i] = 0; a_len[i] = tile0 + i < p.row_tiles ? 0x7fffffffu : 0u; }
    if (RANGED) {
        const int32_t* range = p.tile_range + (int64_t)b * p.row_tiles * 2;
        int lo = 0x7fffffff, hi = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int t = min(tile0 + i, p.row_tiles - 1), l = range[2 * t], e = range[2 * t + 1];
            a_lo[i] = uniform32((uint32_t)l);
            if (a_len[i]) a_len[i] = uniform32((uint32_t)e) - a_lo[i];
            if (e > 0) { lo = min(lo, l); hi = max(hi, e); }
        }
        k_hi = min(k_hi, hi);
        k_lo = max(k_lo, min(lo, hi));
    }
    k_hi = uniform32(k_hi);
    k_lo = uniform32(k_lo);
    int k_next = k_lo + BK * wave;                      // first token of this wave's next stage to request; ranges begin with a block of 128
    const int steps = k_hi > k_next ? (k_hi - k_next + 127) / 128 : 0;

    u32x4 ds[NS][2][2];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) ds[s][i >> 1][i & 1] = u32x4{0u, 0u, 0u, 0u};
    const char* a_ptr = uniform_ptr(reinterpret_cast<const char*>(p.ds + ((int64_t)b * p.Hq + h) * p.ds_bh) +
                                    ((int64_t)(k_lo >> 7) * p.row_tiles + tile0) * 8192 + wave * 2048);
    const uint32_t krow_b = (uint32_t)p.ks.s * 2u;
    const char* b_ptr = uniform_ptr(reinterpret_cast<const char*>(p.k + b * p.ks.b + p.by_G.quotient(h) * p.ks.h) + (int64_t)k_next * krow_b);
    const uint32_t ring = (uint32_t)(uintptr_t)lds + (uint32_t)wave * (NS * STAGE);
    const int b_row = lane / CPR;                       // and RPL further in every load
    // the permutation of a row's chunks depends on its token mod 4 (two tokens to a 256-byte row: mod 4, halved)
    const uint32_t b_chunk = (uint32_t)(((lane % CPR) ^ (LW == 128 ? (lane >> 4) << 2 : ((lane >> 4) & 1) << 2)) & (DH / 8 - 1)) * 16u;
    const uint32_t b_off = (uint32_t)b_row * krow_b + b_chunk;
    auto issue = [&](u32x4 (&to)[2][2], int slot) __attribute__((always_inline)) {
        const uint64_t a = (uint64_t)(uintptr_t)a_ptr;
        const u32x4 srd = {(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, 16384u, 0x00020000u};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t off = (uint32_t)lane * 16u + ((uint32_t)k_next - a_lo[i] < a_len[i] ? 8192u * i : 0x80000000u);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                if (STREAM) asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen offset:%3 nt" : "+v"(to[kk][i]) : "v"(off), "s"(srd), "n"(1024 * kk));
                else asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen offset:%3" : "+v"(to[kk][i]) : "v"(off), "s"(srd), "n"(1024 * kk));
        }
        const int last = k_hi - 1 - k_next;             // rows of K past the last one repeat it: dS^T is zero there
#pragma unroll
        for (int j = 0; j < NKL; ++j) {
            uint32_t off = b_off + (uint32_t)(RPL * j) * krow_b;
            if (last < BK - 1) off = (uint32_t)min(b_row + RPL * j, last) * krow_b + b_chunk;
            dma16(b_ptr, off, ring + slot * STAGE + j * 1024);
        }
        k_next += 128;
        a_ptr += (int64_t)p.row_tiles * 8192;
        b_ptr += (int64_t)128 * krow_b;
    };
    const int r = (lane & 15) >> 2, t = lane & 3, u = (lane >> 4) & 1;
    uint32_t b_rd[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
        b_rd[dt] = (uint32_t)(wave * (NS * STAGE) + (8 * g + r) * ROWB + 64 * (dt ^ (LW == 128 ? r : r >> 1)) + (2 * u + (t >> 1)) * 16 + (t & 1) * 8);
    f32x16 acc[2][NDT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][dt][v] = 0.f;

#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < steps) issue(ds[s], s);
    int k_at = k_lo + BK * wave;
    for (int s0 = 0; s0 < steps; s0 += NS) {
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int s = s0 + i;
            if (s >= steps) break;
            asm volatile("s_cmp_ge_i32 %0, %1\n\ts_cbranch_scc1 LVX_DQ_MORE_%=\n\ts_waitcnt vmcnt(0)\nLVX_DQ_MORE_%=:\n\ts_waitcnt vmcnt(%2)"
                         ::"s"(uniform32(steps - s)), "n"(NS - 1), "n"((NS - 2) * NL) : "memory", "scc");
#pragma unroll
            for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(ds[i][j >> 1][j & 1]));
            wait_lds();         // the stage before has been read
            if (s + NS - 1 < steps) issue(ds[(i + NS - 1) % NS], (i + NS - 1) % NS);
            if (k_at + BK > k_hi) {         // the last stage: tokens past the end count as zeros
#pragma unroll
                for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const int left = k_hi - (k_at + 16 * kk + 8 * g + 2 * w);
                        const uint32_t keep = left >= 2 ? 0xffffffffu : left == 1 ? 0xffffu : 0u;
                        ds[i][kk][0][w] &= keep;
                        ds[i][kk][1][w] &= keep;
                    }
            }
            const char* const st = lds + i * STAGE;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    const bf16x8 kt = lds_operand_tr(reinterpret_cast<const uint16_t*>(st + b_rd[dt] + kk * 16 * ROWB), 4 * LW);
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[j][dt] = E::mfma(kt, as_bf16x8(ds[i][kk][j]), acc[j][dt]);
                }
            k_at += 128;
        }
    }

    // The four sums: chunk c (d = 8 c + 4 g .. + 3 of row l32) of tile j from all waves; wave w adds its half of the chunks of
    // tile w / 2.
    __syncthreads();            // every wave is done with its ring
    char* const sums = lds + lane * 16;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 2 * CW; ++c)
            *reinterpret_cast<f32x4*>(sums + ((wave * 2 + j) * 2 * CW + c) * 1024) =
                f32x4{acc[j][c >> 2][4 * (c & 3)], acc[j][c >> 2][4 * (c & 3) + 1], acc[j][c >> 2][4 * (c & 3) + 2], acc[j][c >> 2][4 * (c & 3) + 3]};
    __syncthreads();
    const int j = wave >> 1, c0 = (wave & 1) * CW, row0 = (tile0 + j) * 32;
    f32x4 x[CW];
#pragma unroll
    for (int c = 0; c < CW; ++c) {
        x[c] = *reinterpret_cast<const f32x4*>(sums + (j * 2 * CW + c0 + c) * 1024);
#pragma unroll
        for (int w = 1; w < 4; ++w) x[c] += *reinterpret_cast<const f32x4*>(sums + ((w * 2 + j) * 2 * CW + c0 + c) * 1024);
    }
    if (p.k_splits > 1) {       // partial tiles, fp32, in this split's slice [B * Hq][DH][rows]: 128 bytes a store
        if (row0 + l32 >= p.rows) return;
        float* const out = p.part + split * p.part_split + (((int64_t)b * p.Hq + h) * DH + 8 * c0 + 4 * g) * p.rows + row0 + l32;
#pragma unroll
        for (int c = 0; c < CW; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) out[(int64_t)(8 * c + e) * p.rows] = x[c][e];
        return;
    }
    __syncthreads();            // the sums have been read
    constexpr int RPS = 64 / CW;                                    // rows per store
    char* const ep = lds + wave * (32 * EP);
#pragma unroll
    for (int c = 0; c < CW; ++c) *reinterpret_cast<u32x2*>(ep + l32 * EP + c * 16 + g * 8) = u32x2{E::pack(x[c][0], x[c][1]), E::pack(x[c][2], x[c][3])};
    wait_lds();
    uint16_t* const out = p.dq + b * p.dqs.b + h * p.dqs.h + (c0 + lane % CW) * 8;
#pragma unroll
    for (int i = 0; i < (32 + RPS - 1) / RPS; ++i) {
        const int row = i * RPS + lane / CW;
        if (row < 32 && row0 + row < p.rows)
            __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(ep + row * EP + (lane % CW) * 16),
                                        reinterpret_cast<u32x4*>(out + (int64_t)(row0 + row) * p.dqs.s));
    }
}

template <int DH, bool F16>
hipError_t launch_dq_t(const DqParams& p, hipStream_t st) {
    const dim3 grid(p.cast_wg + (p.total_wg + 7) / 8 * 8);
    auto go = [&](auto stream, auto ranged) {
        constexpr bool S = decltype(stream)::value, R = decltype(ranged)::value;
        if (p.few) return launch1((dq_few_kernel<DH, F16, S, R>), grid, dim3(256), st, p);
        return launch1((dq_kernel<DH, F16, S, R>), grid, dim3(256), st, p);
    };
    if (p.tile_range) return p.stream ? go(std::true_type{}, std::true_type{}) : go(std::false_type{}, std::true_type{});
    return p.stream ? go(std::true_type{}, std::false_type{}) : go(std::false_type{}, std::false_type{});
}

}  // namespace

hipError_t launch_dq(const DqParams& params, hipStream_t st, const CastSlicesParams* cast) {
    DqParams p = params;
    if (cast) {
        p.cast = *cast;
        p.cast_wg = cast_slices_blocks(*cast);
    }
    if (p.order && (!p.tile_range || p.k_splits > 1 || p.few)) return hipErrorInvalidValue;
    const int group = p.few ? DQ_FEW_TILES : 8;
    const int tiles_m = (p.row_tiles + group - 1) / group, splits = p.k_splits > 1 ? p.k_splits : 1;
    p.total_wg = p.B * p.Hq * tiles_m * splits;
    p.by_splits = divisor(splits);
    p.by_tiles_m = divisor(tiles_m);
    p.by_B = divisor(p.B);
    p.by_Hq = divisor(p.Hq);
    p.by_G = divisor(p.G);
    switch (p.D) {
        case 16: return p.f16 ? launch_dq_t<16, true>(p, st) : launch_dq_t<16, false>(p, st);
        case 32: return p.f16 ? launch_dq_t<32, true>(p, st) : launch_dq_t<32, false>(p, st);
        case 64: return p.f16 ? launch_dq_t<64, true>(p, st) : launch_dq_t<64, false>(p, st);
        case 128: return p.f16 ? launch_dq_t<128, true>(p, st) : launch_dq_t<128, false>(p, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace lvx

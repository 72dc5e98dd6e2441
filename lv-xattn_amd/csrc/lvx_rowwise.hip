// The HBM-bound row-wise kernels of the path: the LSE rescale-merge, the
// backward preprocess (delta = rowsum(O * dO)) and the final fp32 -> bf16
// rounding of an accumulator.  With head_dim 128 a row is 16 lanes x 16 bytes,
// so a 256-thread group streams 16 rows per pass with fully coalesced 256-byte
// row segments; with head_dim 64 / 32 / 16 it is 8 / 4 / 2 lanes and 32 / 64 / 128 rows per pass.
#include "lvx_common.hpp"
#include "lvx_fold.hpp"
#include "lvx_kernels.hpp"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace lvx {

namespace {

// Where the r-th of the rows of all (b, h) is.  Rows are counted in 32 bits: 2^32 of them, 32 bytes each at the least, are
// not in the card's memory twice.
struct RowOf {
    int row, bh, b, h;
    __device__ __forceinline__ RowOf(uint32_t r, const Divisor& by_rows, const Divisor& by_H) {
        uint32_t x, y;
        bh = (int)by_rows.split(r, x);
        b = (int)by_H.split((uint32_t)bh, y);
        row = (int)x;
        h = (int)y;
    }
};

// The block of a kernel that sums what the kernel before it left in parts.  That one deals its (sample, head) pairs, heads
// slowest, to the XCDs in eight contiguous ranges; with the same ranges here the parts are still in the XCD's own L2 (4 MB;
// blocks in order of their number took 7/8 of them from the memory side).  Sixteen rounds of 256 rows x 32 heads x 6404 keys,
// 33 MB of dQ slices and 17 MB of forward parts each: sum 9.0 -> 6.8 us, fold 6.8 -> 6.2; forward and backward 2876 ->
// 2833 us, forward alone 591 -> 586.
__device__ __forceinline__ uint32_t producer_block(uint32_t blocks_per_xcd) {
    return (blockIdx.x & 7) * blocks_per_xcd + (blockIdx.x >> 3);
}

// (o_acc, l_acc) <- merge(acc?, part_0 .. part_{n-1}) for every (b, h, row).  PL lanes share the parts
// of a 16-byte column of a row: with few rows (a token being generated, cut into dozens of key
// ranges) the launch is as long as a thread's chain of loads, so the parts of a row go side by side
// and each thread has the loads of four parts in flight, O beside the LSE it will be weighted by.  PART32: the
// parts are fp32.
template <bool F16, int PL, bool PART32>
__global__ __launch_bounds__(256) void merge_kernel(const MergeParams p) {
    using E = Elt<F16>;
    constexpr int PSH = PL == 4 ? 2 : PL == 2 ? 1 : 0, BATCH = FOLD_BATCH;
    fetch_kernargs<sizeof(MergeParams)>();
    const int nrows = p.row_end - p.row_begin;
    const int64_t idx = (int64_t)producer_block(p.blocks_per_xcd) * 256 + threadIdx.x;
    const int sh = chunk_shift(p.D);
    const int chunk = (int)(idx & ((1 << sh) - 1));
    const int pl = (int)(idx >> sh) & (PL - 1);
    const int64_t r = idx >> (sh + PSH);
    if (r >= (int64_t)p.B * p.Hq * nrows) return;      // the lanes of a row leave together
    uint32_t r_in, b;
    const int h = (int)p.by_B.split(p.by_rows.split((uint32_t)r, r_in), b);
    const int row = p.row_begin + (int)r_in, bh = (int)b * p.Hq + h;

    RowFold sum;
    uint16_t* oa = p.o_acc + b * p.oa.b + h * p.oa.h + (int64_t)row * p.oa.s + chunk * 8;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    float la = -INFINITY;
    u32x4 ua = zero;
    if (p.use_acc && pl == 0) {
        la = p.l_in ? p.l_in[(int64_t)bh * p.l_in_bh + row] : p.l_acc[(int64_t)bh * p.l_acc_bh + row];
        ua = *reinterpret_cast<const u32x4*>(p.o_in ? p.o_in + b * p.oi.b + h * p.oi.h + (int64_t)row * p.oi.s + chunk * 8 : oa);
    }
    const int64_t at = b * p.op.b + h * p.op.h + (int64_t)row * p.op.s + chunk * 8;
    const uint16_t* op = p.o_part + at;
    const float* op32 = reinterpret_cast<const float*>(p.o_part) + at;
    const float* lp = p.l_part + (int64_t)bh * p.l_part_bh + row;
    for (int i = pl; i < p.nparts; i += PL * BATCH) {
        float l[BATCH];
        u32x4 u[BATCH], u2[PART32 ? BATCH : 1];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            const int part = i + k * PL;
            const bool ok = part < p.nparts;
            l[k] = ok ? lp[part * p.l_part_stride] : -INFINITY;
            if constexpr (PART32) {
                u[k] = ldg16(op32 + part * p.o_part_stride, ok);
                u2[k] = ldg16(op32 + part * p.o_part_stride + 4, ok);
            } else {
                u[k] = ldg16(op + part * p.o_part_stride, ok);
            }
        }
        sum.add(l, [&](int k, float (&f)[8]) {
            if constexpr (PART32) {
#pragma unroll
                for (int j = 0; j < 4; ++j) { f[j] = __uint_as_float(u[k][j]); f[4 + j] = __uint_as_float(u2[k][j]); }
            } else {
                unpack8<E>(u[k], f);
            }
        });
    }
    if (p.use_acc) {
        const float l[BATCH] = {la, -INFINITY, -INFINITY, -INFINITY};
        sum.add(l, [&](int k, float (&f)[8]) { unpack8<E>(k ? zero : ua, f); });
    }
#pragma unroll
    for (int o = 1; o < PL; o <<= 1) {                  // the lanes that share a row's parts
        const int d = o << sh;
        RowFold other;
        other.m = __shfl_xor(sum.m, d);
        other.den = __shfl_xor(sum.den, d);
#pragma unroll
        for (int j = 0; j < 8; ++j) other.out[j] = __shfl_xor(sum.out[j], d);
        sum.join(other);
    }
    if (pl != 0) return;
    *reinterpret_cast<u32x4*>(oa) = sum.result<E>();
    if (chunk == 0) p.l_acc[(int64_t)bh * p.l_acc_bh + row] = sum.lse();
}

// The same for one part folded into the accumulator (what lvx_merge does every round), two rows
// per thread: every load of both rows is issued before the first use, so a thread keeps
// 64 + 8 bytes in flight.  780 bytes per (row, head).
template <bool F16>
__global__ __launch_bounds__(256) void merge_pair_kernel(const MergeParams p) {
    using E = Elt<F16>;
    fetch_kernargs<sizeof(MergeParams)>();
    const int nrows = p.row_end - p.row_begin;
    const int64_t total = (int64_t)p.B * p.Hq * nrows;
    const int64_t half = (total + 1) / 2;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int sh = chunk_shift(p.D);
    const int chunk = (int)(idx & ((1 << sh) - 1));
    const int64_t r0 = idx >> sh;
    if (r0 >= half) return;
    int64_t rr[2] = {r0, r0 + half};
    const bool ok1 = rr[1] < total;
    if (!ok1) rr[1] = r0;
    uint16_t* oa[2];
    const uint16_t* op[2];
    float* la_p[2];
    float la[2], lb[2];
    u32x4 ua[2], ub[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const RowOf at_row((uint32_t)rr[k], p.by_rows, p.by_Hq);
        const int row = p.row_begin + at_row.row, bh = at_row.bh, b = at_row.b, h = at_row.h;
        oa[k] = p.o_acc + b * p.oa.b + h * p.oa.h + (int64_t)row * p.oa.s + chunk * 8;
        op[k] = p.o_part + b * p.op.b + h * p.op.h + (int64_t)row * p.op.s + chunk * 8;
        la_p[k] = p.l_acc + (int64_t)bh * p.l_acc_bh + row;
        la[k] = *la_p[k];
        lb[k] = p.l_part[(int64_t)bh * p.l_part_bh + row];
        ua[k] = *reinterpret_cast<const u32x4*>(oa[k]);
        ub[k] = *reinterpret_cast<const u32x4*>(op[k]);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if (k == 1 && !ok1) break;
        const float m = fmaxf(la[k], lb[k]);
        const float ms = (m == -INFINITY) ? 0.f : m;
        const float wa = __expf(la[k] - ms), wb = __expf(lb[k] - ms);
        const float den = wa + wb;
        const float inv = den > 0.f ? 1.f / den : 0.f;
        // a side with weight 0 may hold anything (it saw no key, or nothing was folded in yet)
        const float ca = wa * inv, cb = wb * inv;
        float fa[8], fb[8];
        unpack8<E>(ua[k], fa);
        unpack8<E>(ub[k], fb);
        u32x4 u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float x0 = (ca > 0.f ? fa[2 * j] * ca : 0.f) + (cb > 0.f ? fb[2 * j] * cb : 0.f);
            const float x1 = (ca > 0.f ? fa[2 * j + 1] * ca : 0.f) + (cb > 0.f ? fb[2 * j + 1] * cb : 0.f);
            u[j] = E::pack(x0, x1);
        }
        *reinterpret_cast<u32x4*>(oa[k]) = u;
        if (chunk == 0) *la_p[k] = den > 0.f ? ms + __logf(den) : -INFINITY;
    }
}

// A row's sum of products, of the eight of each of its 1 << sh lanes.
template <class E>
__device__ __forceinline__ float row_dot(u32x4 a, u32x4 b, int sh) {
    float x[8], y[8], s = 0.f;
    unpack8<E>(a, x);
    unpack8<E>(b, y);
#pragma unroll
    for (int j = 0; j < 8; ++j) s = fmaf(x[j], y[j], s);
    if (sh >= 4) s += __shfl_xor(s, 8);
    if (sh >= 3) s += __shfl_xor(s, 4);
    if (sh >= 2) s += __shfl_xor(s, 2);
    return s + __shfl_xor(s, 1);
}

// delta = rowsum(O * dO): head_dim / 8 lanes x 16 bytes per row and tensor, two rows per thread with all
// four loads issued before the first use.  516 bytes per (row, head).
template <bool F16>
__global__ __launch_bounds__(256) void preprocess_kernel(const PreParams p) {
    using E = Elt<F16>;
    fetch_kernargs<sizeof(PreParams)>();
    const int nrows = p.row_end - p.row_begin;
    const int64_t total = (int64_t)p.B * p.Hq * nrows;
    const int64_t half = (total + 1) / 2;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int sh = chunk_shift(p.D);
    const int chunk = (int)(idx & ((1 << sh) - 1));
    const int64_t r0 = idx >> sh;
    const bool ok0 = r0 < half;                         // the lanes of a row share the flags
    const bool ok1 = ok0 && r0 + half < total;
    const int64_t rr[2] = {ok0 ? r0 : 0, ok1 ? r0 + half : 0};
    u32x4 uo[2], ud[2];
    float* out[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const RowOf at_row((uint32_t)rr[k], p.by_rows, p.by_Hq);
        const int row = p.row_begin + at_row.row, bh = at_row.bh, b = at_row.b, h = at_row.h;
        const bool ok = k ? ok1 : ok0;
        uo[k] = ldg16(p.o + b * p.os.b + h * p.os.h + (int64_t)row * p.os.s + chunk * 8, ok);
        ud[k] = ldg16(p.dout + b * p.ds.b + h * p.ds.h + (int64_t)row * p.ds.s + chunk * 8, ok);
        out[k] = p.delta + (int64_t)bh * p.Lq + row;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float s = row_dot<E>(uo[k], ud[k], sh);
        if ((k ? ok1 : ok0) && chunk == 0) *out[k] = s;
    }
}

// The i-th shared block's number in the list of token blocks, or -1 if the last XCD has no such block.
__device__ __forceinline__ int shared_block(const SharedBlocks& s, int i) {
    const int per = s.blocks_per_xcd - s.whole;
    const int blk0 = i / per * s.blocks_per_xcd, at = s.whole + i % per, nblk = min(s.blocks_per_xcd, s.n_blocks - blk0);
    if (at >= nblk) return -1;
    return blk0 + at;
}

// A row's key interval, (INT_MAX, 0) where it sees nothing or lies past the window.
__device__ __forceinline__ void row_interval(const LiveParams& p, int b, int kv_len, int r, int& lo, int& hi) {
    const int64_t at = (int64_t)b * p.Lq + min(r, p.row_end - 1);
    lo = max(p.kv_start[at], 0);
    hi = min(p.kv_end[at], kv_len);
    if (r >= p.row_end || hi <= lo) { lo = INT_MAX; hi = 0; }
}
__device__ __forceinline__ int len_of(const LiveParams& p, int b) { return p.kv_len ? min(p.kv_len[b], p.Lkv) : p.Lkv; }
// The hull of the intervals of a lane's 32, in whole token blocks.
__device__ __forceinline__ void hull_of_32(int& lo, int& hi) {
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
        lo = min(lo, __shfl_xor(lo, o));
        hi = max(hi, __shfl_xor(hi, o));
    }
    lo = hi > 0 ? (lo / 128) * 128 : 0;
    hi = (hi + 127) / 128 * 128;
}

// One thread per row: the hulls of the row tiles' key intervals in whole token blocks.  i: work-group, of hull_blocks.
__host__ __device__ __forceinline__ int hull_blocks(const LiveParams& p) { return (p.n_tiles + 7) / 8 * p.B; }
__device__ __forceinline__ void tile_hulls(const LiveParams& p, int i) {
    const int per = (p.n_tiles + 7) / 8, b = i / per, tile = (i - b * per) * 8 + (threadIdx.x >> 5);
    int lo, hi;
    row_interval(p, b, len_of(p, b), p.row_begin + tile * 32 + (threadIdx.x & 31), lo, hi);
    hull_of_32(lo, hi);
    if ((threadIdx.x & 31) == 0 && tile < p.n_tiles) {
        int32_t* h = p.tile_hull + ((int64_t)b * p.n_tiles + tile) * 2;
        h[0] = lo;
        h[1] = hi;
    }
}

// One wave: the runs of consecutive row tiles whose hull (h, [n_tiles][2]) holds token block kblk.  Where there are more than
// four, the two the narrowest gap apart become one, so that the three widest gaps are left out.
__device__ __forceinline__ void live_runs(const LiveParams& p, const int32_t* h, int b, int kblk) {
    const int lane = threadIdx.x & 63, kvb = kblk * 128;
    int first[4] = {0, 0, 0, 0}, end[4] = {0, 0, 0, 0}, nr = 0, last_end = -1;
    for (int t0 = 0; t0 < p.n_tiles; t0 += 64) {
        const int32_t* const ht = h + min(t0 + lane, p.n_tiles - 1) * 2;
        uint64_t live = __builtin_amdgcn_ballot_w64(t0 + lane < p.n_tiles && ht[0] <= kvb && kvb < ht[1]);
        while (live) {
            const int bit = __builtin_ctzll(live), s = t0 + bit;
            const uint64_t gaps = ~(live >> bit);
            const int n = min(gaps ? __builtin_ctzll(gaps) : 64, 64 - bit), e = s + n;
            live &= n == 64 ? 0 : ~(((uint64_t{1} << n) - 1) << bit);
            const bool apart = s != last_end, append = apart && nr < 4;
            if (apart && !append) {
                int width = s - end[3], at = 3;
#pragma unroll
                for (int i = 2; i >= 0; --i)
                    if (first[i + 1] - end[i] < width) { width = first[i + 1] - end[i]; at = i; }
#pragma unroll
                for (int i = 0; i < 3; ++i) {   // close gap `at`: the runs on its sides become one, the later ones move up
                    if (i >= at) end[i] = end[i + 1];
                    if (i > at) first[i] = first[i + 1];
                }
                if (at < 3) first[3] = s;
            }
            if (append) ++nr;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i == nr - 1) { if (append) first[i] = s; end[i] = e; }
            last_end = e;
        }
    }
    if (lane < 8) {
        int x = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (lane == 2 * i && i < nr) x = first[i];
            if (lane == 2 * i + 1 && i < nr) x = end[i] - first[i];
        }
        p.live_runs[((int64_t)b * p.n_kv_blocks + kblk) * 8 + lane] = x;
    }
}

// Group i of n is as many places behind the first as there are longer ones and, before it, equally long ones.
__device__ __forceinline__ void rank_group(const LiveParams& p, const int* len, int i, int n) {
    const int mine = len[i];
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += (len[j] > mine || (len[j] == mine && j < i)) ? 1 : 0;
    p.order[rank] = i;
}

// The same tables without one launch waiting for another, where there are few row tiles: four token blocks of a sample to a
// work-group, which takes the hulls of the sample's tiles itself (a few loads per thread, all in flight, at most MAX_LIVE_TILES
// tiles in all samples); the sample's first writes them down as well, and one more work-group takes the hulls of the groups
// and ranks them.
__host__ __device__ __forceinline__ int live_blocks(const LiveParams& p) {
    return (p.plan.entries ? 8 : 0) + (p.n_kv_blocks + 3) / 4 * p.B + (p.order ? 1 : 0);
}

// The hulls of the tiles of samples [b0, b0 + nb) into LDS, by the whole work-group, 2 AHEAD loads per thread in flight.
template <int AHEAD>
__device__ __forceinline__ void hulls_to_lds(const LiveParams& p, int b0, int nb, int32_t* hull) {
    const int n = nb * p.n_tiles;
    for (int t0 = 0; t0 < n; t0 += 8 * AHEAD) {
        int lo[AHEAD], hi[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            uint32_t tile;
            const int b = b0 + (int)p.by_tiles.split((uint32_t)min(t0 + 8 * k + (int)(threadIdx.x >> 5), n - 1), tile);
            row_interval(p, b, len_of(p, b), p.row_begin + (int)tile * 32 + (int)(threadIdx.x & 31), lo[k], hi[k]);
        }
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            const int t = t0 + 8 * k + (int)(threadIdx.x >> 5);
            hull_of_32(lo[k], hi[k]);
            if ((threadIdx.x & 31) == 0 && t < n) { hull[2 * t] = lo[k]; hull[2 * t + 1] = hi[k]; }
        }
    }
}

// See PlanParams; one work-group, for XCD x.  hull: of the tiles of all samples.  The longest blocks, as many as make whole rounds of the XCD's CUs, stay whole.  The ranges of
// the others are priced as choose_bwd_cut does, in steps (about a microsecond): six for what a work-group spends outside them, and for
// writing the slices and adding them up 8 and 0.3 per slice.
__device__ __forceinline__ void plan_xcd(const LiveParams& p, int x, const int32_t* hull) {
    __shared__ __attribute__((aligned(16))) int key[MAX_PLANNED_BLOCKS];
    __shared__ int sorted[MAX_PLANNED_BLOCKS];          // steps << 8 | block
    const PlanParams& q = p.plan;
    const int tid = threadIdx.x;
    const int blk0 = x * q.blocks_per_xcd, n = max(0, min(q.blocks_per_xcd, q.n_blocks - blk0));
    static_assert(MAX_PLANNED_BLOCKS == 256, "a thread to a block, eight bits of a key");
    key[tid] = -1;
    __syncthreads();
    const int sh = n <= 64 ? 2 : n <= 128 ? 1 : 0, j = tid >> sh;       // threads to a block
    int tiles = 0;
    if (j < n) {
        const int id = blk0 + j, kvb = id % p.n_kv_blocks * 128, b = id / p.n_kv_blocks % p.B;
        const int32_t* const h = hull + 2 * b * p.n_tiles;
#pragma unroll 4
        for (int t = tid & ((1 << sh) - 1); t < p.n_tiles; t += 1 << sh) tiles += h[2 * t] <= kvb && kvb < h[2 * t + 1] ? 1 : 0;
    }
    for (int o = 1; o < 1 << sh; o <<= 1) tiles += __shfl_xor(tiles, o);
    if (j < n) key[j] = tiles * q.G << 8 | j;
    __syncthreads();
    const int mine = key[tid];
    int rank = 0;
#pragma unroll 2
    for (int k = 0; k < (n + 3) / 4; ++k) {
        const u32x4 other = reinterpret_cast<const u32x4*>(key)[k];
#pragma unroll
        for (int e = 0; e < 4; ++e) rank += (int)other[e] > mine ? 1 : 0;
    }
    if (tid < n) sorted[rank] = mine;
    const int n_live = __syncthreads_count(mine > 255);     // of one step and more
    const int whole = n_live / q.cus * q.cus, rest = n_live - whole;
    const float longest = rest ? (float)(sorted[whole] >> 8) : 0.f;
    int S = 1;
    float best = longest + 6.f;
    for (int s = 2; s <= 8 && longest >= (float)(MIN_PLANNED_RANGE * s) && rest * (s - 1) <= q.slots - q.blocks_per_xcd && rest * s <= q.slices; ++s) {
        const float cost = (float)((rest * s + q.cus - 1) / q.cus) * (longest / (float)s + 6.f) + 8.f + 0.3f * (float)(rest * s);
        if (cost < best) { best = cost; S = s; }
    }
    const int ranges = S > 1 ? rest * S : 0, first_dead = n_live + (ranges ? ranges - rest : 0);
    uint32_t* const out = q.entries + (int64_t)x * q.slots * PLAN_ENTRY;
    for (int l = tid; l < q.slots; l += 256) {
        uint32_t e = ~0u, slice = 0;
        const int r = l - whole;
        if (r >= 0 && r < ranges) {
            e = (uint32_t)(sorted[whole + r / S] & 255) | (uint32_t)S << 16 | (uint32_t)(r % S) << 24;
            slice = (uint32_t)(x * q.slices + r - r % S);
        } else {
            const int at = l < first_dead ? l : l - first_dead + n_live;
            if (at < n) e = (uint32_t)(sorted[at] & 255) | 1u << 16;
        }
        out[l * PLAN_ENTRY] = e;
        out[l * PLAN_ENTRY + 1] = slice;
    }
    for (int j = tid; j < q.shared_max; j += 256) {
        uint32_t* const e = q.shared + (int64_t)(x * q.shared_max + j) * SHARED_ENTRY;
        const bool cut = ranges && j < rest;
        e[0] = cut ? (uint32_t)(blk0 + (sorted[whole + j] & 255)) : 0u;
        e[1] = cut ? (uint32_t)S : 0u;
        e[2] = (uint32_t)(x * q.slices + j * S);
    }
}

__device__ __forceinline__ void live_tables(const LiveParams& p, int i) {
    __shared__ int32_t hull[MAX_LIVE_TILES * 2];
    // the plans first, they take longest
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, per = (p.n_kv_blocks + 3) / 4, plans = p.plan.entries ? 8 : 0;
    const int b = i < plans ? 0 : (i - plans) / per;
    if (b >= p.B) {
        const int n = p.B * p.n_groups;
        int* const len = hull;
        for (int j = wave; j < n; j += 4) {
            const int gb = j / p.n_groups, r0 = p.row_begin + (j - gb * p.n_groups) * (LIVE_GROUP * 32) + lane, kv_len = len_of(p, gb);
            int lo[4], hi[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) row_interval(p, gb, kv_len, r0 + 64 * k, lo[k], hi[k]);
            int l = min(min(lo[0], lo[1]), min(lo[2], lo[3])), h = max(max(hi[0], hi[1]), max(hi[2], hi[3]));
            l = min(l, __shfl_xor(l, 32));
            h = max(h, __shfl_xor(h, 32));
            hull_of_32(l, h);
            if (lane == 0) len[j] = h - l;
        }
        __syncthreads();
        if ((int)threadIdx.x < n) rank_group(p, len, threadIdx.x, n);
        return;
    }
    // (one copy of it: what a launch as short as this waits for is its instructions on their way from memory)
    hulls_to_lds<8>(p, b, i < plans ? p.B : 1, hull);
    __syncthreads();
    if (i < plans) {
        plan_xcd(p, i, hull);
        return;
    }
    i -= plans;
    const int kblk = (i - b * per) * 4 + wave;
    if (kblk < p.n_kv_blocks) live_runs(p, hull, b, kblk);
    if (i != b * per) return;
    for (int k = threadIdx.x; k < 2 * p.n_tiles; k += 256) p.tile_hull[(int64_t)b * p.n_tiles * 2 + k] = hull[k];
}

// LSE and delta of the window, re-expressed once for the backward kernel: the
// exponent offset LSE * log2(e), +inf for rows that saw no key or lie past the
// window (so that P = exp2(x - inf) = 0 there), and delta * scale (0 past the
// window), grouped per 32-row tile so that one 256-byte load fetches a tile's lot.
struct MetaRow {
    const MetaParams& p;
    int begin, end, n_tiles;                // of this window
    __device__ __forceinline__ explicit MetaRow(const MetaParams& params) : p(params) {
        begin = p.row_begin + (int)blockIdx.y * p.round_rows;
        end = min(begin + p.round_rows, p.row_end);
        n_tiles = (end - begin + 31) / 32;  // a last window may be shorter
    }
    __device__ __forceinline__ void write(int64_t bh, uint32_t r, float l, float d) const {
        float* o = p.out + blockIdx.y * p.round_out + (bh * n_tiles + (r >> 5)) * 64 + (r & 31);
        o[0] = (l == -INFINITY) ? INFINITY : l * 1.4426950408889634f;
        o[32] = d * p.scale;
    }
};

// FROM_O: delta = rowsum(O * dO) is formed here, the loads and sums of preprocess_kernel, whose launch and whose 4 bytes a row there
// and back it saves.  Bound by reading O and dO.  us alone, preprocess_kernel, records and tables of a mask in launches of their own ->
// in one: 4096 rows x 32 heads 12.0 + 5.4 -> 16.0, 2048 x 32 of 64 5.6 + 6.9 -> 7.1, 2 x 3000 x 32 with a mask 16.1 + 5.1 + 5.6 -> 18.2,
// 1024 x 16 with one 5.0 + 5.0 + 5.6 -> 5.3 (forward and backward 231 -> 225).
template <bool FROM_O, bool F16>
__global__ __launch_bounds__(256) void bwd_meta_kernel(const MetaParams p) {
    fetch_kernargs<sizeof(MetaParams)>();
    // With an interval mask the first blocks write its tables, or where there are many row tiles their hulls
    if ((int)blockIdx.x < p.table_blocks) {
        if (blockIdx.y) return;
        if (p.tables) live_tables(p.live, (int)blockIdx.x);
        else tile_hulls(p.live, (int)blockIdx.x);
        return;
    }
    // the last blocks of the launch zero the scratches (stores rather than hipMemsetAsync, so
    // that callers may capture the stream)
    if ((int)blockIdx.x >= p.meta_end) {
        const int z = (int)blockIdx.x - p.meta_end;
        const int blk = shared_block(p.sb, z / SHARE_PARTS);
        if (blk < 0) return;
        const int kblk = blk % p.sb.n_kv_blocks, bh = blk / p.sb.n_kv_blocks, zb = bh % p.sb.B, hk = bh / p.sb.B;
        const int sh = chunk_shift(p.sb.D) + 1;         // 16-byte chunks of a row of floats
        const int64_t half = (int64_t)p.sb.B * p.sb.Lkv * p.sb.Hkv * p.sb.D;
        for (int i = threadIdx.x; i < (SHARE_ROWS << sh); i += 256) {
            const int token = kblk * 128 + z % SHARE_PARTS * SHARE_ROWS + (i >> sh);
            if (token >= p.sb.Lkv) return;
            float* d = p.scratch + (((int64_t)zb * p.sb.Lkv + token) * p.sb.Hkv + hk) * p.sb.D + (i & ((1 << sh) - 1)) * 4;
            *reinterpret_cast<u32x4*>(d) = u32x4{0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4*>(d + half) = u32x4{0u, 0u, 0u, 0u};
        }
        return;
    }
    const MetaRow rec(p);
    const int64_t total = (int64_t)p.B * p.Hq * p.n_tiles * 32;
    const int64_t idx = (int64_t)((int)blockIdx.x - p.table_blocks) * 256 + threadIdx.x;
    if constexpr (!FROM_O) {
        if (idx >= total) return;
        uint32_t r;
        const int64_t bh = p.by_rows.split((uint32_t)idx, r);
        if ((int)(r >> 5) >= rec.n_tiles) return;
        const int row = rec.begin + (int)r;
        const bool ok = row < rec.end;
        rec.write(bh, r, ok ? p.lse[bh * p.Lq + row] : -INFINITY, ok ? p.delta[bh * p.Lq + row] : 0.f);
    } else {
        using E = Elt<F16>;
        const int sh = chunk_shift(p.D), chunk = (int)(idx & ((1 << sh) - 1));
        const int64_t half = total / 2, r0 = idx >> sh;             // total: whole tiles
        if (r0 >= half) return;                                     // (the lanes of a row leave together)
        u32x4 uo[2], ud[2];
        float l[2];
        uint32_t r[2];
        int64_t bh[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const RowOf at((uint32_t)(r0 + k * half), p.by_rows, p.by_Hq);
            r[k] = (uint32_t)at.row;
            bh[k] = at.bh;
            const int row = rec.begin + at.row;
            const bool ok = row < rec.end;
            uo[k] = ldg16(p.o + at.b * p.os.b + at.h * p.os.h + (int64_t)row * p.os.s + chunk * 8, ok);
            ud[k] = ldg16(p.dout + at.b * p.ds.b + at.h * p.ds.h + (int64_t)row * p.ds.s + chunk * 8, ok);
            l[k] = ok ? p.lse[bh[k] * p.Lq + row] : -INFINITY;
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float s = row_dot<E>(uo[k], ud[k], sh);
            if (chunk == 0 && (int)(r[k] >> 5) < rec.n_tiles) rec.write(bh[k], r[k], l[k], s);
        }
    }
}

// Per (b, text row) the first and one-past-last key whose bias is not -inf, over all heads the bias distinguishes.  An
// empty row gets (0, 0).  WAVES: waves that share a row, 1 or 4; BATCH: loads of 16 bytes a thread has in flight (see
// launch_bias_hull).  Bound by reading the bias, once; a wave reads long rows from both ends inwards, as far as these hide
// something (most biases hide neither, and nothing between them matters then).
template <int WAVES, int BATCH>
__global__ __launch_bounds__(256) void bias_hull_kernel(const BiasHullParams p) {
    constexpr int STEP = 4 * 64 * WAVES;                    // keys one load of the waves covers
    fetch_kernargs<sizeof(BiasHullParams)>();
    const uint32_t rows = (uint32_t)p.B * (uint32_t)p.Lq, wave = uniform32(threadIdx.x >> 6);
    const int lane = WAVES == 1 ? threadIdx.x & 63 : threadIdx.x;
    for (uint32_t rw = WAVES == 1 ? blockIdx.x * 4 + wave : blockIdx.x; rw < rows; rw += gridDim.x * (4 / WAVES)) {
        uint32_t row;
        const uint32_t b = p.by_Lq.split(rw, row);
        int lo = INT_MAX, hi = 0;
        const auto see = [&](const f32x4& v, int k) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (k + j < p.Lkv && !(v[j] == -INFINITY)) { lo = min(lo, k + j); hi = max(hi, k + j + 1); }
        };
        for (int h = 0; h < p.heads; ++h) {
            const float* br = p.bias + b * p.bias_b + h * p.bias_h + (int64_t)row * p.bias_r;
            if (WAVES == 1 && BATCH == 4 && p.Lkv > BATCH * STEP) {
                int first = 0, end = (p.Lkv + 3) & ~3;          // the keys that are left
                bool low = true, high = true;                   // nothing seen below them, above them
                while (first < end && (low || high)) {
                    const int n = low ? high ? (BATCH + 1) / 2 : BATCH : 0;
                    f32x4 v[BATCH];
                    int k[BATCH];
#pragma unroll
                    for (int i = 0; i < BATCH; ++i) {
                        k[i] = max(4 * lane + (i < n ? first + STEP * i : end - STEP * (i - n + 1)), 0);
                        v[i] = *reinterpret_cast<const f32x4*>(br + min(k[i], (p.Lkv - 1) & ~3));
                    }
#pragma unroll
                    for (int i = 0; i < BATCH; ++i) see(v[i], k[i]);
                    first += STEP * n;
                    end -= STEP * (BATCH - n);
                    low = low && __builtin_amdgcn_ballot_w64(lo < first) == 0;
                    high = high && __builtin_amdgcn_ballot_w64(hi > end) == 0;
                }
                continue;
            }
            for (int k0 = 4 * lane; k0 < p.Lkv; k0 += BATCH * STEP) {
                f32x4 v[BATCH];
#pragma unroll
                for (int i = 0; i < BATCH; ++i)
                    v[i] = *reinterpret_cast<const f32x4*>(br + min(k0 + i * STEP, (p.Lkv - 1) & ~3));
#pragma unroll
                for (int i = 0; i < BATCH; ++i) see(v[i], k0 + i * STEP);
            }
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            lo = min(lo, __shfl_xor(lo, o));
            hi = max(hi, __shfl_xor(hi, o));
        }
        if constexpr (WAVES > 1) {
            __shared__ int red[WAVES][2];
            __syncthreads();        // the row before has been read
            if ((threadIdx.x & 63) == 0) { red[wave][0] = lo; red[wave][1] = hi; }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < WAVES; ++w) { lo = min(lo, red[w][0]); hi = max(hi, red[w][1]); }
        }
        if (lane == 0) {
            p.kv_start[rw] = hi > 0 ? lo : 0;
            p.kv_end[rw] = hi;
        }
    }
}

// One wave per (b, text row): sets *p.flag when an entry of the row's bias inside [kv_start, kv_end)
// is not exactly zero, i.e. when the bias is more than the interval mask its hull describes.
__global__ __launch_bounds__(256) void bias_interval_kernel(const BiasHullParams p) {
    const int64_t rw = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (rw >= (int64_t)p.B * p.Lq) return;
    const int b = (int)(rw / p.Lq), row = (int)(rw % p.Lq);
    const int lo = max(p.kv_start[rw], 0), hi = min(p.kv_end[rw], p.Lkv);
    bool other = false;
    for (int h = 0; h < p.heads; ++h) {
        const float* br = p.bias + b * p.bias_b + h * p.bias_h + (int64_t)row * p.bias_r;
        for (int k0 = (lo & ~3) + 4 * lane; k0 < hi; k0 += 256) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(br + k0);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (k0 + j >= lo && k0 + j < hi && !(v[j] == 0.f)) other = true;
        }
    }
    if (__builtin_amdgcn_ballot_w64(other) != 0 && lane == 0) atomicOr(p.flag, 1);
}

// One work-group per (b, text row) of a mask in the model's own type: first and one-past-last key that is not
// masked (an entry above -30000), and whether the row is that interval and nothing else - every
// entry inside it exactly 0, at least one.  Reads the mask once, 2 bytes per (row, key), where turning
// it into an fp32 bias and looking for the hull of that took ten launches and 16 bytes (2 x 300 rows x
// 6404 keys: 75 us, this: 8).  Up to four 8-byte words of a thread are in flight, and a wave asks for none behind the row's
// last (us back to back in bf16, so / one in flight / four whatever the row's length: 4 x 1 rows x 6404 keys 3.8 / 4.3 /
// 3.9, x 400 2.3 / 2.3 / 2.9, 4 x 1024 x 801 6.6 / 6.6 / 9.2, x 6404 14.4 / 14.9 / 15.4).  Rows start on any element, so an 8-byte load
// may begin before the row or end behind it; it stays inside the 8-byte word that holds an element of the row.
template <typename T>
__global__ __launch_bounds__(256) void mask_interval_kernel(const MaskIntervalParams p) {
    constexpr int EPW = 8 / sizeof(T);                  // elements per 8-byte word
    __shared__ int red[4][4];
    fetch_kernargs<sizeof(MaskIntervalParams)>();
    uint32_t row;
    const uint32_t b = p.by_Lq.split(blockIdx.x, row);
    const T* r = static_cast<const T*>(p.mask) + b * p.stride_b + (int64_t)row * p.stride_r;
    const int skew = (int)((reinterpret_cast<uintptr_t>(r) & 7) / sizeof(T));       // elements of the first word before the row
    const uint2* words = reinterpret_cast<const uint2*>(r - skew);
    int lo = INT_MAX, hi = 0, n = 0, other = 0;
    const int lane = threadIdx.x & 63;
    const int n_words = (p.Lkv + skew + EPW - 1) / EPW;
    constexpr int BATCH = 4;                            // words of a thread in flight
    for (int w0 = uniform32((int)threadIdx.x & ~63); w0 < n_words; w0 += BATCH * 256) {    // this wave's first word
      uint2 us[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i)
        if (w0 + i * 256 < n_words) us[i] = words[min(w0 + i * 256 + lane, n_words - 1)];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        if (w0 + i * 256 >= n_words) break;
        const int w = w0 + i * 256 + lane;
        const uint2 u = us[i];
#pragma unroll
        for (int e = 0; e < EPW; ++e) {
            const int key = w * EPW + e - skew;
            float x;
            if constexpr (sizeof(T) == 4) x = __uint_as_float(e ? u.y : u.x);
            else {
                const uint32_t pair = e < 2 ? u.x : u.y;
                if constexpr (std::is_same<T, _Float16>::value) x = e & 1 ? Elt<true>::hi(pair) : Elt<true>::lo(pair);
                else x = e & 1 ? bf16_hi(pair) : bf16_lo(pair);
            }
            if (key >= 0 && key < p.Lkv && !(x <= -30000.f)) {
                lo = min(lo, key);
                hi = max(hi, key + 1);
                ++n;
                other |= !(x == 0.f);
            }
        }
      }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        lo = min(lo, __shfl_xor(lo, o));
        hi = max(hi, __shfl_xor(hi, o));
        n += __shfl_xor(n, o);
        other |= __shfl_xor(other, o);
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { red[wave][0] = lo; red[wave][1] = hi; red[wave][2] = n; red[wave][3] = other; }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < 4; ++w) {
        lo = min(lo, red[w][0]);
        hi = max(hi, red[w][1]);
        n += red[w][2];
        other |= red[w][3];
    }
    const bool interval = n > 0 && hi - lo == n && !other;
    p.kv_start[blockIdx.x] = interval ? lo : -1;
    p.kv_end[blockIdx.x] = interval ? hi : 0;
}

__global__ __launch_bounds__(256) void bwd_hull_kernel(const LiveParams p) { tile_hulls(p, blockIdx.x); }

// One wave per (token block, b): its runs.
// Blocks past those (b == 0 only) rank the groups of row tiles by the length of their hull, one thread per group.
__global__ __launch_bounds__(64) void bwd_live_kernel(const LiveParams p) {
    const int lane = threadIdx.x;
    if ((int)blockIdx.x >= p.n_kv_blocks) {
        __shared__ int len[MAX_RANKED_GROUPS];
        const int n = p.B * p.n_groups, i = ((int)blockIdx.x - p.n_kv_blocks) * 64 + lane;
        if (blockIdx.y != 0) return;
        for (int j = lane; j < n; j += 64) {
            const int b = j / p.n_groups, t0 = (j - b * p.n_groups) * LIVE_GROUP;
            const int32_t* h = p.tile_hull + (int64_t)b * p.n_tiles * 2;
            int lo = INT_MAX, hi = 0;
#pragma unroll
            for (int k = 0; k < LIVE_GROUP; ++k) {
                const int t = min(t0 + k, p.n_tiles - 1);
                if (h[2 * t + 1] > 0) { lo = min(lo, h[2 * t]); hi = max(hi, h[2 * t + 1]); }
            }
            len[j] = max(0, hi - lo);
        }
        __syncthreads();
        if (i < n) rank_group(p, len, i, n);
        return;
    }
    live_runs(p, p.tile_hull + (int64_t)blockIdx.y * p.n_tiles * 2, blockIdx.y, blockIdx.x);
}

template <bool F16>
__global__ __launch_bounds__(256) void cast_kernel(const CastParams p) {
    using E = Elt<F16>;
    fetch_kernargs<sizeof(CastParams)>();
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int sh = chunk_shift(p.D);
    const int Dh = 8 << sh;
    const int chunk = (int)(idx & ((1 << sh) - 1));
    const int64_t r = idx >> sh;
    if (r >= (int64_t)p.B * p.H * p.L) return;
    const RowOf at_row((uint32_t)r, p.by_L, p.by_H);
    const int row = at_row.row, b = at_row.b, h = at_row.h;
    const f32x4* s = reinterpret_cast<const f32x4*>(p.src + r * Dh + chunk * 8);
    const f32x4 a = s[0], c = s[1];
    u32x4 u;
    u[0] = E::pack(a[0], a[1]);
    u[1] = E::pack(a[2], a[3]);
    u[2] = E::pack(c[0], c[1]);
    u[3] = E::pack(c[2], c[3]);
    *reinterpret_cast<u32x4*>(p.dst + b * p.ds.b + h * p.ds.h + (int64_t)row * p.ds.s + chunk * 8) = u;
}

// The shared token blocks of the scratch (SHARE_PARTS work-groups each) into dK and dV.  Only those blocks are
// zeroed before and rounded after: in a layer with 2 x 6404 tokens and 1023 rows 48 of 816, the layer's
// step 1928 -> 1888 us.
template <bool F16>
__global__ __launch_bounds__(256) void cast_shared_kernel(const CastSharedParams p) {
    using E = Elt<F16>;
    const int blk = shared_block(p.sb, (int)blockIdx.x / SHARE_PARTS);
    if (blk < 0) return;
    const int kblk = blk % p.sb.n_kv_blocks, bh = blk / p.sb.n_kv_blocks, b = bh % p.sb.B, hk = bh / p.sb.B;
    const int sh = chunk_shift(p.sb.D);
    const int64_t half = (int64_t)p.sb.B * p.sb.Lkv * p.sb.Hkv * p.sb.D;
    for (int i = threadIdx.x; i < (SHARE_ROWS << sh); i += 256) {
        const int token = kblk * 128 + (int)(blockIdx.x % SHARE_PARTS) * SHARE_ROWS + (i >> sh), chunk = i & ((1 << sh) - 1);
        if (token >= p.sb.Lkv) return;
        const float* s = p.scratch + (((int64_t)b * p.sb.Lkv + token) * p.sb.Hkv + hk) * p.sb.D + chunk * 8;
        const f32x4 k0 = *reinterpret_cast<const f32x4*>(s), k1 = *reinterpret_cast<const f32x4*>(s + 4);
        const f32x4 v0 = *reinterpret_cast<const f32x4*>(s + half), v1 = *reinterpret_cast<const f32x4*>(s + half + 4);
        const u32x4 ku = {E::pack(k0[0], k0[1]), E::pack(k0[2], k0[3]), E::pack(k1[0], k1[1]), E::pack(k1[2], k1[3])};
        const u32x4 vu = {E::pack(v0[0], v0[1]), E::pack(v0[2], v0[3]), E::pack(v1[0], v1[1]), E::pack(v1[2], v1[3])};
        *reinterpret_cast<u32x4*>(p.dk + b * p.dks.b + hk * p.dks.h + (int64_t)token * p.dks.s + chunk * 8) = ku;
        *reinterpret_cast<u32x4*>(p.dv + b * p.dvs.b + hk * p.dvs.h + (int64_t)token * p.dvs.s + chunk * 8) = vu;
    }
}

template <bool F16>
__global__ __launch_bounds__(256) void cast_slices_kernel(const CastSlicesParams p) { cast_slices<F16>(p, blockIdx.x); }

// cast_kernel from a transposed source (cast_t).
template <bool F16>
__global__ __launch_bounds__(256) void cast_t_kernel(const CastParams p) {
    fetch_kernargs<sizeof(CastParams)>();
    cast_t<F16>(p, (int64_t)producer_block(p.blocks_per_xcd) * 256 + threadIdx.x);
}

// Backward of y = w * bf16(x * r) over 128-wide rows: with xh = x * r and gg = dy * w,
//   dx = r * (gg - xh * mean(gg * xh)),   dw += sum over rows of dy * bf16(xh).
// 16 lanes per row (8 columns each); a thread keeps the dw partial sums of its 8 columns over the rows
// it visits, the block folds them through LDS and adds them with 128 atomics.  All blocks add to the
// same 128 floats, which takes 0.2 ns an addition: with 2048 blocks that was the kernel (57 us on 102464
// rows, whose 79 MB take 15 us to move), so there is one block of 1024 threads per CU, each thread
// with the loads of two rows in flight: 19 us.
constexpr int NORM_THREADS = 1024, NORM_ROWS = NORM_THREADS / 16, NORM_BLOCKS = 256;

template <bool F16>
__global__ __launch_bounds__(NORM_THREADS) void norm_bwd_kernel(const NormBwdParams p) {
    using E = Elt<F16>;
    __shared__ float fold[NORM_ROWS][16][8];
    const int sub = threadIdx.x & 15, grp = threadIdx.x >> 4;
    const int64_t nrows = (int64_t)p.M * p.heads;
    const u32x4 wu = *reinterpret_cast<const u32x4*>(p.w + sub * 8);
    float w[8], dwp[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) { w[2 * j] = E::lo(wu[j]); w[2 * j + 1] = E::hi(wu[j]); }
#pragma unroll
    for (int j = 0; j < 8; ++j) dwp[j] = 0.f;
    const int64_t stride = (int64_t)gridDim.x * NORM_ROWS;
    for (int64_t row0 = (int64_t)blockIdx.x * NORM_ROWS + grp; row0 < nrows; row0 += 2 * stride) {
        u32x4 du[2], xu[2];
        float r[2];
        uint16_t* out[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const bool ok = row0 + k * stride < nrows;          // the lanes of a row agree
            const int64_t row = ok ? row0 + k * stride : row0;
            const int64_t m = row / p.heads;
            const int h = (int)(row % p.heads);
            du[k] = ldg16(p.dy + m * p.ldy + h * 128 + sub * 8, ok);    // zero: adds nothing to dw
            xu[k] = ldg16(p.x + m * p.ldx + h * 128 + sub * 8, ok);
            r[k] = p.rstd[row];
            out[k] = ok ? p.dx + m * p.lddx + h * 128 + sub * 8 : nullptr;
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float gg[8], xh[8], c = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float d0 = E::lo(du[k][j]), d1 = E::hi(du[k][j]);
                xh[2 * j] = E::lo(xu[k][j]) * r[k];
                xh[2 * j + 1] = E::hi(xu[k][j]) * r[k];
                gg[2 * j] = d0 * w[2 * j];
                gg[2 * j + 1] = d1 * w[2 * j + 1];
                const uint32_t xb = E::pack(xh[2 * j], xh[2 * j + 1]);
                dwp[2 * j] = fmaf(d0, E::lo(xb), dwp[2 * j]);
                dwp[2 * j + 1] = fmaf(d1, E::hi(xb), dwp[2 * j + 1]);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) c = fmaf(gg[j], xh[j], c);
            c = sum16(c) * (1.f / 128.f);
            u32x4 u;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                u[j] = E::pack(r[k] * (gg[2 * j] - xh[2 * j] * c), r[k] * (gg[2 * j + 1] - xh[2 * j + 1] * c));
            if (out[k]) *reinterpret_cast<u32x4*>(out[k]) = u;
        }
    }
    if (!p.dw) return;
#pragma unroll
    for (int j = 0; j < 8; ++j) fold[grp][sub][j] = dwp[j];
    __syncthreads();
    if (threadIdx.x < 128) {
        const int s2 = threadIdx.x >> 3, j = threadIdx.x & 7;
        float t = 0.f;
#pragma unroll 8
        for (int gi = 0; gi < NORM_ROWS; ++gi) t += fold[gi][s2][j];
        unsafeAtomicAdd(p.dw + threadIdx.x, t);
    }
}

inline uint32_t per_xcd(int64_t threads) { return (uint32_t)((threads + 8 * 256 - 1) / (8 * 256)); }
inline int blocks_for(int64_t rows) { return (int)((rows * 16 + 255) / 256); }

}  // namespace

hipError_t launch_merge(const MergeParams& params, hipStream_t st) {
    MergeParams p = params;
    const int64_t rows = (int64_t)p.B * p.Hq * (p.row_end - p.row_begin);
    if (rows == 0) return hipSuccess;
    p.by_rows = divisor(p.row_end - p.row_begin);
    p.by_Hq = divisor(p.Hq);
    if (p.nparts == 1 && p.use_acc && !p.o_in) {
        const dim3 grid(blocks_for((rows + 1) / 2));
        if (p.f16) return launch1(merge_pair_kernel<true>, grid, dim3(256), st, p);
        return launch1(merge_pair_kernel<false>, grid, dim3(256), st, p);
    }
    const int pl = fold_chains(p.nparts, rows);
    p.by_B = divisor(p.B);
    p.blocks_per_xcd = per_xcd((rows * pl << chunk_shift(p.D)));
    const dim3 grid(8 * p.blocks_per_xcd);
    auto go = [&](auto f16, auto part32) {
        constexpr bool F16 = decltype(f16)::value;
        constexpr bool PART32 = decltype(part32)::value;
        if (pl == 4) return launch1(merge_kernel<F16, 4, PART32>, grid, dim3(256), st, p);
        if (pl == 2) return launch1(merge_kernel<F16, 2, PART32>, grid, dim3(256), st, p);
        return launch1(merge_kernel<F16, 1, PART32>, grid, dim3(256), st, p);
    };
    if (p.part_f32) return p.f16 ? go(std::true_type{}, std::true_type{}) : go(std::false_type{}, std::true_type{});
    return p.f16 ? go(std::true_type{}, std::false_type{}) : go(std::false_type{}, std::false_type{});
}

hipError_t launch_preprocess(const PreParams& params, hipStream_t st) {
    PreParams p = params;
    const int64_t rows = (int64_t)p.B * p.Hq * (p.row_end - p.row_begin);
    if (rows == 0) return hipSuccess;
    p.by_rows = divisor(p.row_end - p.row_begin);
    p.by_Hq = divisor(p.Hq);
    if (p.f16) return launch1(preprocess_kernel<true>, dim3(blocks_for((rows + 1) / 2)), dim3(256), st, p);
    else return launch1(preprocess_kernel<false>, dim3(blocks_for((rows + 1) / 2)), dim3(256), st, p);
}

hipError_t launch_bwd_meta(const MetaParams& p0, hipStream_t st, const LiveParams* live) {
    MetaParams p = p0;
    if (live && live->n_tiles > 0 && live->B > 0) {
        p.live = *live;
        p.live.by_tiles = divisor(live->n_tiles);
        p.tables = live_in_one(*live);
        p.table_blocks = p.tables ? live_blocks(*live) : hull_blocks(*live);
    }
    const int64_t rows = p.out ? (int64_t)p.B * p.Hq * p.n_tiles * 32 : 0, n = p.o ? rows / 2 << chunk_shift(p.D) : rows;
    const int zero_blocks = p.scratch ? 8 * (p.sb.blocks_per_xcd - p.sb.whole) * SHARE_PARTS : 0;
    if (n == 0 && zero_blocks == 0 && p.table_blocks == 0) return hipSuccess;
    p.meta_end = p.table_blocks + (int)((n + 255) / 256);
    p.by_rows = divisor(std::max(1, p.n_tiles * 32));
    p.by_Hq = divisor(std::max(1, p.Hq));
    const dim3 grid((unsigned)(p.meta_end + zero_blocks), std::max(1, p.rounds));
    if (!p.o) return launch1(bwd_meta_kernel<false, false>, grid, dim3(256), st, p);
    if (p.f16) return launch1(bwd_meta_kernel<true, true>, grid, dim3(256), st, p);
    return launch1(bwd_meta_kernel<true, false>, grid, dim3(256), st, p);
}

hipError_t launch_bwd_live(const LiveParams& p, hipStream_t st, bool has_hulls) {
    if (p.B <= 0 || p.n_groups <= 0 || p.n_kv_blocks <= 0) return hipSuccess;
    if (live_in_one(p)) return has_hulls ? hipSuccess : launch_bwd_meta(MetaParams{}, st, &p);
    if (!has_hulls) {
        const hipError_t e = launch1(bwd_hull_kernel, dim3(hull_blocks(p)), dim3(256), st, p);
        if (e != hipSuccess) return e;
    }
    const int rank_blocks = p.order ? (p.B * p.n_groups + 63) / 64 : 0;
    return launch1(bwd_live_kernel, dim3(p.n_kv_blocks + rank_blocks, p.B), dim3(64), st, p);
}

// A wave to a row, with as many loads in flight as a row of so many keys has, up to four; a work-group to a row where rows
// are long and there are too few of them to keep the chip reading.  us, a wave to a row / a work-group to a row, four loads:
// 1024 rows x 1000 keys 2.5 / 3.5, x 2500 3.3 / 3.6, x 4096 3.9 / 3.7, x 6404 5.3 / 4.9; 2048 x 4096 4.8 / 5.2; 1 x 1300 2.26
// / 2.13, 1 x 13000 5.7 / 3.1.  16384 x 400 with one, two and four loads 6.2, 5.9, 7.3 / 17.4; a wave to a row with one load
// took 5.0 at 1024 x 4096 and 20.8 (10.7 with four) at 1024 x 13000.
// From both ends inwards, nothing hidden / half of the row at one end, before -> now: 1024 x 4096 3.5 (a work-group to a row) -> 2.5 / 3.4,
// 2048 x 4096 4.8 -> 2.8 / 4.1, 1024 x 6404 4.6 -> 2.5 / 3.9, 1024 x 13000 9.6 -> 2.5 / 6.5; 256 x 4096 would go 2.6 -> 2.45 / 3.3 and 64 x 13000
// 3.5 -> 2.4 / 5.
hipError_t launch_bias_hull(const BiasHullParams& params, hipStream_t st) {
    BiasHullParams p = params;
    const int64_t rows = (int64_t)p.B * p.Lq;
    if (rows == 0) return hipSuccess;
    p.by_Lq = divisor(p.Lq);
    const dim3 by_wave((unsigned)std::min<int64_t>((rows + 3) / 4, 1 << 20));
    if (p.Lkv <= 256) return launch1((bias_hull_kernel<1, 1>), by_wave, dim3(256), st, p);
    if (p.Lkv <= 512) return launch1((bias_hull_kernel<1, 2>), by_wave, dim3(256), st, p);
    if (p.Lkv <= 1024 || rows > std::min(512, p.Lkv / 4)) return launch1((bias_hull_kernel<1, 4>), by_wave, dim3(256), st, p);
    return launch1((bias_hull_kernel<4, 4>), dim3((unsigned)rows), dim3(256), st, p);
}

hipError_t launch_mask_intervals(const MaskIntervalParams& params, hipStream_t st) {
    MaskIntervalParams p = params;
    p.by_Lq = divisor(p.Lq);
    const dim3 grid((unsigned)((int64_t)p.B * p.Lq));
    if (p.type == 1) return launch1(mask_interval_kernel<uint16_t>, grid, dim3(256), st, p);
    if (p.type == 2) return launch1(mask_interval_kernel<_Float16>, grid, dim3(256), st, p);
    return launch1(mask_interval_kernel<float>, grid, dim3(256), st, p);
}

hipError_t launch_bias_interval(const BiasHullParams& p, hipStream_t st) {
    const int64_t rows = (int64_t)p.B * p.Lq;
    if (rows == 0) return hipSuccess;
    return launch1(bias_interval_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), st, p);
}

hipError_t launch_norm_bwd(const NormBwdParams& p, hipStream_t st) {
    const int64_t rows = (int64_t)p.M * p.heads;
    if (rows == 0) return hipSuccess;
    const dim3 grid((unsigned)std::min<int64_t>((rows + NORM_ROWS - 1) / NORM_ROWS, NORM_BLOCKS));
    if (p.f16) return launch1(norm_bwd_kernel<true>, grid, dim3(NORM_THREADS), st, p);
    else return launch1(norm_bwd_kernel<false>, grid, dim3(NORM_THREADS), st, p);
}

hipError_t launch_cast_shared(const CastSharedParams& p, hipStream_t st) {
    const dim3 grid(8 * (p.sb.blocks_per_xcd - p.sb.whole) * SHARE_PARTS);
    if (grid.x == 0) return hipSuccess;
    if (p.f16) return launch1(cast_shared_kernel<true>, grid, dim3(256), st, p);
    return launch1(cast_shared_kernel<false>, grid, dim3(256), st, p);
}

hipError_t launch_cast_slices(const CastSlicesParams& p, hipStream_t st) {
    const dim3 grid(cast_slices_blocks(p));
    if (grid.x == 0) return hipSuccess;
    if (p.f16) return launch1(cast_slices_kernel<true>, grid, dim3(256), st, p);
    return launch1(cast_slices_kernel<false>, grid, dim3(256), st, p);
}

// For cast_t by work-groups of so many threads.
hipError_t plan_cast_t(CastParams& p, int threads) {
    const int64_t rows = (int64_t)p.B * p.H * p.L;
    if (rows * 16 > UINT32_MAX) return hipErrorInvalidValue;    // 256 rows of dQ at most per CU
    p.by_L = divisor(p.L);
    p.by_B = divisor(p.B);
    p.blocks_per_xcd = (uint32_t)((((rows << chunk_shift(p.D)) + threads - 1) / threads + 7) / 8);
    return hipSuccess;
}

hipError_t launch_cast(const CastParams& params, hipStream_t st) {
    CastParams p = params;
    const int64_t rows = (int64_t)p.B * p.H * p.L;
    if (rows == 0) return hipSuccess;
    p.by_L = divisor(p.L);
    p.by_H = divisor(p.H);
    const dim3 grid(blocks_for(rows));
    if (p.transposed) {
        const hipError_t e = plan_cast_t(p, 256);
        if (e != hipSuccess) return e;
        const dim3 grid(8 * p.blocks_per_xcd);
        if (p.f16) return launch1(cast_t_kernel<true>, grid, dim3(256), st, p);
        else return launch1(cast_t_kernel<false>, grid, dim3(256), st, p);
    } else {
        if (p.f16) return launch1(cast_kernel<true>, grid, dim3(256), st, p);
        else return launch1(cast_kernel<false>, grid, dim3(256), st, p);
    }
}

}  // namespace lvx

// The fold of partial results of attention rows, a 16-byte column of a row at a time: what merge_kernel does with
// the parts of a launch, and what the forward does with those of the launch before it.  Both take the parts in the same
// order and the same groups, so that a row's bits do not depend on which of them folded it.
#pragma once
#include "lvx_common.hpp"
#include "lvx_fold_rule.hpp"
#include "lvx_kernels.hpp"

namespace lvx {

constexpr int FOLD_BATCH = 4;       // parts that join at once; chain c of n takes parts c, c + n, c + 2 n ..

struct RowFold {
    float m = -INFINITY, den = 0.f, out[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // Folds the parts (l[k], values by part(k, f)) in; a part with weight 0 may hold anything (it saw no key, or nothing
    // had been folded into the accumulator yet), one with weight NaN makes the row NaN
    template <class Part>
    __device__ __forceinline__ void add(const float (&l)[FOLD_BATCH], Part&& part) {
        float mn = m;
#pragma unroll
        for (int k = 0; k < FOLD_BATCH; ++k) mn = fmaxf(mn, l[k]);
        const float ms = (mn == -INFINITY) ? 0.f : mn;
        const float keep = __expf(m - ms);
        den *= keep;
#pragma unroll
        for (int j = 0; j < 8; ++j) out[j] *= keep;
#pragma unroll
        for (int k = 0; k < FOLD_BATCH; ++k) {
            const float w = __expf(l[k] - ms);
            den += w;
            float f[8];
            part(k, f);
#pragma unroll
            for (int j = 0; j < 8; ++j) out[j] = w != 0.f ? fmaf(f[j], w, out[j]) : out[j];
        }
        m = mn;
    }
    __device__ __forceinline__ void join(const RowFold& o) {
        const float mn = fmaxf(m, o.m), ms = (mn == -INFINITY) ? 0.f : mn;
        const float w1 = __expf(m - ms), w2 = __expf(o.m - ms);
        den = fmaf(den, w1, o.den * w2);
#pragma unroll
        for (int j = 0; j < 8; ++j) out[j] = fmaf(out[j], w1, o.out[j] * w2);
        m = mn;
    }
    template <class E>
    __device__ __forceinline__ u32x4 result() const {
        const float inv = den > 0.f ? 1.f / den : 0.f;
        u32x4 u;
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] = E::pack(out[2 * j] * inv, out[2 * j + 1] * inv);
        return u;
    }
    __device__ __forceinline__ float lse() const { return den > 0.f ? m + __logf(den) : -INFINITY; }
};

// log2 of the 16-byte chunks (lanes) per row
__host__ __device__ __forceinline__ int chunk_shift(int head_dim) {
    return head_dim == 64 ? 3 : head_dim == 32 ? 2 : head_dim == 16 ? 1 : 4;
}

// Rounds eight values of a row of the fp32 source [B*H][D][L], or of the sum of several such: thread `idx` of the launch.  Adjacent
// threads take adjacent rows, so the eight strided reads of a thread are coalesced across the wave.
template <bool F16>
__device__ __forceinline__ void cast_t(const CastParams& p, int64_t idx) {
    using E = Elt<F16>;
    const int sh = chunk_shift(p.D);
    const int Dh = 8 << sh;
    if (idx >= ((int64_t)p.B * p.H * p.L << sh)) return;
    uint32_t row, b;       // plan_cast_t checks that a thread's number fits 32 bits
    const uint32_t col = p.by_L.split((uint32_t)idx, row);      // a chunk of an (h, b)
    const int chunk = (int)(col & ((1u << sh) - 1));
    const int h = (int)p.by_B.split(col >> sh, b), bh = (int)b * p.H + h;
    const float* s = p.src + ((int64_t)bh * Dh + chunk * 8) * p.L + row;
    float a[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = s[(int64_t)j * p.L];
    for (int k = 1; k < p.nsum; ++k) {
        s += p.sum_stride;
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] += s[(int64_t)j * p.L];
    }
    u32x4 u;
#pragma unroll
    for (int j = 0; j < 4; ++j) u[j] = E::pack(a[2 * j], a[2 * j + 1]);
    *reinterpret_cast<u32x4*>(p.dst + b * p.ds.b + h * p.ds.h + (int64_t)row * p.ds.s + chunk * 8) = u;
}

// A token block of the scratch is zeroed and rounded by SHARE_PARTS work-groups of SHARE_ROWS tokens each.
constexpr int SHARE_ROWS = 128 / SHARE_PARTS;

// Work-group i of 256 threads.  The blocks that have been cut, SHARE_PARTS work-groups each: their slices added in the order of their ranges and rounded.  All blocks of
// an XCD's list are its own again, whose L2 may still hold the slices.
template <bool F16>
__device__ __forceinline__ void cast_slices(const CastSlicesParams& p, uint32_t i) {
    using E = Elt<F16>;
    const int xcd = i % 8, part = (int)(i / 8 % SHARE_PARTS), j = (int)(i / (8 * SHARE_PARTS));
    int blk, S, slice;
    if (p.shared) {
        const uint32_t* const e = p.shared + (int64_t)(xcd * p.shared_max + j) * SHARED_ENTRY;
        blk = (int)e[0];
        S = (int)e[1];
        slice = (int)e[2];
        if (S == 0) return;
    } else {
        const bool second = j >= p.mid;
        S = second ? p.splits2 : p.splits;
        slice = xcd * p.slices_per_xcd + (second ? p.mid * p.splits + (j - p.mid) * S : j * S);
        blk = xcd * p.blocks_per_xcd + p.whole + j;
        if (blk >= min((xcd + 1) * p.blocks_per_xcd, p.n_blocks)) return;
    }
    const int kblk = blk % p.n_kv_blocks, bh = blk / p.n_kv_blocks, b = bh % p.B, hk = bh / p.B;
    const int sh = chunk_shift(p.D);
    const int64_t half = (int64_t)128 * p.D;
    const float* const src = p.slices + (int64_t)slice * 2 * half;
    for (int k = threadIdx.x; k < (SHARE_ROWS << sh); k += 256) {
        const int r = part * SHARE_ROWS + (k >> sh), token = kblk * 128 + r, chunk = k & ((1 << sh) - 1);
        if (token >= p.Lkv) return;
        const float* s = src + (int64_t)r * p.D + chunk * 8;
        f32x4 x[4] = {};
#pragma unroll 4
        for (int n = 0; n < S; ++n, s += 2 * half) {
            x[0] += *reinterpret_cast<const f32x4*>(s);
            x[1] += *reinterpret_cast<const f32x4*>(s + 4);
            x[2] += *reinterpret_cast<const f32x4*>(s + half);
            x[3] += *reinterpret_cast<const f32x4*>(s + half + 4);
        }
        const u32x4 ku = {E::pack(x[0][0], x[0][1]), E::pack(x[0][2], x[0][3]), E::pack(x[1][0], x[1][1]), E::pack(x[1][2], x[1][3])};
        const u32x4 vu = {E::pack(x[2][0], x[2][1]), E::pack(x[2][2], x[2][3]), E::pack(x[3][0], x[3][1]), E::pack(x[3][2], x[3][3])};
        *reinterpret_cast<u32x4*>(p.dk + b * p.dks.b + hk * p.dks.h + (int64_t)token * p.dks.s + chunk * 8) = ku;
        *reinterpret_cast<u32x4*>(p.dv + b * p.dvs.b + hk * p.dvs.h + (int64_t)token * p.dvs.s + chunk * 8) = vu;
    }
}

template <class E>
__device__ __forceinline__ void unpack8(u32x4 u, float f[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f[2 * j] = E::lo(u[j]);
        f[2 * j + 1] = E::hi(u[j]);
    }
}

}  // namespace lvx

// The fold of partial results of attention rows, a 16-byte column of a row at a time: what merge_kernel does with
// the parts of a launch, and what the forward does with those of the launch before it.  Both take the parts in the same
// order and the same groups, so that a row's bits do not depend on which of them folded it.
#pragma once
#include "lvx_common.hpp"

namespace lvx {

// Lanes (of merge_kernel; chains of fold_before) that share the parts of a row: as many as the parts need, four parts each,
// and the chip has room for.
__host__ __device__ inline int fold_chains(int nparts, int64_t rows) {
    return nparts > 8 && rows < 16384 ? 4 : nparts > 4 && rows < 32768 ? 2 : 1;
}

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

template <class E>
__device__ __forceinline__ void unpack8(u32x4 u, float f[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f[2 * j] = E::lo(u[j]);
        f[2 * j + 1] = E::hi(u[j]);
    }
}

}  // namespace lvx

// Internal launch interface between the C-ABI layer (lvx_api.hip) and the
// kernel translation units.  All sizes have been validated by the caller.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lvx {

// Queues kernel(p) and returns that launch's own error code.  The thread's sticky "last error"
// (which may hold an unrelated component's earlier failure) is neither read nor cleared.
template <typename P>
inline hipError_t launch1(void (*kernel)(P), dim3 grid, dim3 block, hipStream_t st, const P& p) {
    P arg = p;
    void* args[] = {&arg};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, args, 0, st);
}

// CUs of the device that is current (the one the caller's stream belongs to), asked for once per device.
int cu_count();

struct Strides3 {
    int64_t b, h, s;
};

// Which forward kernel: a wave owns 32 rows of a head (heads of 16 and 32, dense bias), 64 rows and its
// SIMD (head dimensions 128 and 64), or a share of the keys for up to 32 (row, head) pairs at once.
enum FwdForm { FWD_PLAIN = 0, FWD_WIDE = 1, FWD_FEW = 2 };

// Division of work-group numbers by something the host knows: a product and a correction instead of the forty
// instructions of an integer division.  floor((2^32 - 1) / d) times x / 2^32 is x / d or one less.
struct Divisor {
    uint32_t d, m;
    __host__ __device__ uint32_t split(uint32_t x, uint32_t& rest) const {
        uint32_t q = (uint32_t)((uint64_t)x * m >> 32);
        rest = x - q * d;
        if (rest >= d) { ++q; rest -= d; }
        return q;
    }
    __host__ __device__ uint32_t quotient(uint32_t x) const { uint32_t rest; return split(x, rest); }
};
inline Divisor divisor(int d) { return Divisor{(uint32_t)d, 0xffffffffu / (uint32_t)d}; }

// The parts of one launch that the next one folds on its way (16-bit parts; wide form).  Null part: none.
struct FwdFold {
    const uint16_t* part;      // [nparts][B * Hq][rows][D]
    const float* l_part;       // [nparts][B * Hq][rows]
    uint16_t* o;               // the result, of the folded window's first row (l: absolute rows, Lq to a (b, h))
    float* l;
    const uint16_t* acc;       // incoming accumulator, indexed like o and l, or null
    const float* l_acc;
    Strides3 os, as;
    int nparts, rows, row_begin;
    // filled in by launch_fwd
    int chains;                // see fold_chains; more than two do not ride
    uint32_t per_wg;           // 16-byte chunks that a work-group folds, whole rows
    Divisor by_rows;
};

struct FwdParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* o;               // float* with o_f32
    float* lse;
    Strides3 qs, ks, vs, os;
    int64_t o_split_stride;    // elements between the partial O of two key splits
    int64_t lse_split_stride;  // floats between the partial LSE of two key splits
    int64_t lse_bh_stride;     // floats between two (b, h) rows of LSE
    const int32_t* kv_len;
    const int32_t* kv_start;
    const int32_t* kv_end;
    const float* bias;         // dense additive bias or nullptr; element strides below
    int64_t bias_b, bias_h, bias_r;
    int B, Hq, Hkv, Lq, Lkv;
    int D;                     // head dimension: 16, 32, 64 or 128
    int G;                     // q heads per kv head
    int HG;                    // q heads a work-group covers (one per wave)
    int RS;                    // row sub-tiles a work-group covers per head
    int form;                  // FwdForm
    int row_begin, row_end;
    int n_row_tiles, n_head_groups, nsplit, split_len, total_wg;
    float scale, scale_log2e;
    int f16;                   // element type of q, k, v, o: 0 bf16, 1 fp16
    int o_f32;                 // 1: o (the parts of a launch with key splits) is fp32
    // Form for few rows: not null, and the key ranges' work-groups leave their fp32 parts, [nsplit][B * Hq][rows][D] and
    // [nsplit][B * Hq][rows], here; the last of a kv head folds them into o and lse, which are then the result's
    float* part;
    float* l_part;
    // filled in by launch_fwd: divisors by n_row_tiles, nsplit, B, G and G / HG
    Divisor by_row_tiles, by_splits, by_B, by_G, by_head_groups;
};

// A launch that also folds the parts of the one before it: arguments that no other launch fills, copies or fetches.
struct FwdFoldParams : FwdParams {
    FwdFold fold;
};

struct MergeParams {
    uint16_t* o_acc;
    float* l_acc;
    const uint16_t* o_part;    // const float* with part_f32
    const float* l_part;
    Strides3 oa, op;
    int64_t o_part_stride;     // elements between consecutive partials
    int64_t l_part_stride;     // floats between consecutive partials
    int64_t l_acc_bh, l_part_bh;
    int nparts;
    int use_acc;               // 1: fold into the existing accumulator, 0: overwrite
    // with use_acc and several parts: where the accumulator is read from when it is not
    // (o_acc, l_acc) itself, which then only receive the result (null: in place)
    const uint16_t* o_in;
    const float* l_in;
    Strides3 oi;
    int64_t l_in_bh;
    int B, Hq, Lq, row_begin, row_end;
    int f16;
    int D;                     // head dimension: 16, 32, 64 or 128 (0 reads as 128)
    int part_f32;              // 1: the parts are fp32 (not for one part folded into an accumulator)
    Divisor by_rows, by_Hq, by_B;   // filled in by launch_merge: rows of the window, q heads, samples
    uint32_t blocks_per_xcd;        // and a share of the grid
};

// Per text row the hull of the keys a dense bias leaves visible (entries other than -inf).
struct BiasHullParams {
    const float* bias;
    int64_t bias_b, bias_h, bias_r;
    int32_t* kv_start;         // [B, Lq]: written by the hull kernel, read by the interval test
    int32_t* kv_end;           // [B, Lq]
    int B, heads, Lq, Lkv;     // heads: 1 (bias broadcast over heads) or Hq
    Divisor by_Lq;             // filled in by launch_bias_hull, for its kernel
    int32_t* flag;             // interval test only: set to 1 when the bias is not 0 everywhere inside the hull
};
// Per text row of an additive mask [B][Lq][Lkv] (type: LVX_BF16, LVX_F16 or 0 for fp32; element strides
// stride_b, stride_r) the interval of keys it leaves visible, where that is all it says.
struct MaskIntervalParams {
    const void* mask;
    int64_t stride_b, stride_r;
    int type;
    int32_t* kv_start;         // [B, Lq]; -1 for a row that is more than an interval
    int32_t* kv_end;           // [B, Lq]
    int B, Lq, Lkv;
    Divisor by_Lq;             // filled in by launch_mask_intervals
};
hipError_t launch_mask_intervals(const MaskIntervalParams& p, hipStream_t st);
hipError_t launch_bias_hull(const BiasHullParams& p, hipStream_t st);
hipError_t launch_bias_interval(const BiasHullParams& p, hipStream_t st);

struct PreParams {
    const uint16_t* o;
    const uint16_t* dout;
    float* delta;
    Strides3 os, ds;
    int B, Hq, Lq, row_begin, row_end;
    int f16;
    int D;                     // head dimension: 16, 32, 64 or 128 (0 reads as 128)
    Divisor by_rows, by_Hq;    // filled in by launch_preprocess
};

struct CastParams {
    const float* src;
    uint16_t* dst;
    Strides3 ds;
    int B, H, L;
    int transposed;   // 0: src is [B*H][L][D]; 1: src is [B*H][D][L]
    int nsum;         // transposed only: the result is the sum of nsum such sources (0 or 1: one),
    int64_t sum_stride;   // sum_stride floats apart
    int f16;          // destination type: 0 bf16, 1 fp16
    int D;            // head dimension: 16, 32, 64 or 128 (0 reads as 128)
    Divisor by_L, by_H, by_B;       // filled in by launch_cast
    uint32_t blocks_per_xcd;        // and a share of the grid
};

struct BwdParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    const uint16_t* dout;
    const float* meta;         // per (b, h, 32-row tile): 32 x LSE*log2(e) (+inf for dead rows), 32 x delta*scale
    uint16_t* ds_ws;           // dS^T workspace [B*Hq][token blocks][row tiles][16 groups of tokens][32 rows][8 tokens]
    int64_t ws_ld;             // elements per token block (row tiles * 4096)
    int64_t ws_bh;             // elements per (b, h) slab
    int ds_stream;             // 1: dS^T is stored with streaming stores (see lvx_bwd)
    void* dk;
    void* dv;
    Strides3 qs, ks, vs, dos, dks, dvs;
    const int32_t* kv_len;
    const int32_t* kv_start;
    const int32_t* kv_end;
    const float* bias;         // dense additive bias or nullptr; element strides below
    int64_t bias_b, bias_h, bias_r;
    int B, Hq, Hkv, Lq, Lkv, G;
    int D;                     // head dimension: 16, 32, 64 or 128
    int row_begin, row_end;
    int n_kv_blocks;
    int n_blocks;              // token blocks of all (b, kv head): B * Hkv * n_kv_blocks
    int blocks_per_xcd;        // ceil(n_blocks / 8): the token blocks an XCD's work-groups take
    int whole_blocks;          // of an XCD's blocks, the first so many get one work-group each (0 .. blocks_per_xcd),
    int mid_blocks, q_splits;  // the next mid_blocks are shared by q_splits work-groups each, every one taking a range of steps,
    int q_splits2;             // and the others by q_splits2 (>= 1) work-groups each
    int dkv_mode;              // 0: store 16-bit, 1: fp32 +=, 2: fp32 atomic += (the shared blocks, not with slices)
    // mode 2: where and how the work-group of a block it owns alone writes (whole_mode 0 or 1)
    void* dk_whole;
    void* dv_whole;
    Strides3 dks_whole, dvs_whole;
    int whole_mode;
    float scale, scale_log2e;
    // Interval masks: the 32-row tiles each token block has to visit (the others see none of
    // its tokens) as up to 4 runs of consecutive tiles, live_runs[(b * n_kv_blocks + block) * 8
    // + 2 i + {0, 1}] = first tile and number of tiles of run i (0 tiles: unused).  Null: every tile.
    const int32_t* live_runs;
    // Not null: which block and range a work-group takes, in place of whole_blocks and the rest (see PlanParams)
    const uint32_t* plan;
    // Not null: a range of a block that has several leaves fp32 sums in a slice of its own, [dK, dV][128 tokens][D]: those of an XCD
    // in the order of its work-groups (with a plan: where it says)
    float* slices;
    int per_xcd;               // entries of the plan, or slices, of an XCD
    int f16;                   // element type of q, k, v, dout, the dS^T workspace and (mode 0) dk, dv
    Divisor by_splits, by_splits2, by_kv_blocks, by_B;     // filled in by launch_bwd
    // and the work-groups that are the token blocks' (a multiple of 8): any past them sum the slices of dQ of the window before
    int own_wg;
    CastParams dq_before;
};

// How the token blocks of a launch with an interval mask are handed to work-groups, where there are at least two of them to a CU.  Their
// lengths are known on the device only, where one work-group per XCD sorts the XCD's blocks: the longest, as many
// as fill whole rounds of its CUs, get a work-group each, the others are cut into ranges of steps, and those nobody sees come last.  A range
// leaves fp32 sums in a slice of its own, [dK, dV][128 tokens][D], and cast_slices_kernel adds and rounds them.
// 2 x 3000 rows that see the image before them (77 blocks of 180 to 368 steps on 32 CUs: 602 steps until the last CU ends, 512 with 13
// cut in two, by a count of steps): bwd_kernel 620 -> 579 us, what the launches before and after it take 19 -> 33, forward and
// backward 1057 -> 1037.  (More CUs at work run at a lower clock.  Whole blocks chosen by simulating which CU is free when, to 512
// steps instead of 552, gave the same kernel and took 20 us longer to plan.)  Others of 500 blocks and more 0 to -6 %.
// Entry l of XCD x: the block's number in the XCD's list | ranges << 16 | range << 24, and the slice of the block's first range; ~0: none.
constexpr int MAX_PLANNED_BLOCKS = 256;         // of an XCD; with more rounds than eight there is little left to even out
constexpr int MIN_PLANNED_RANGE = 24;           // steps: shorter ranges are all ramp
constexpr int PLAN_ENTRY = 2, SHARED_ENTRY = 4;     // words; of a shared block: its number, ranges (0: no such block), slice, unused
struct PlanParams {
    uint32_t* entries;         // out: [8][slots][PLAN_ENTRY]; null: no plan
    uint32_t* shared;          // out: [8][shared_max][SHARED_ENTRY]
    int slots, cus;            // entries and CUs of an XCD
    int shared_max, slices;    // most blocks of an XCD that are cut, most slices (slices x * slices + ..)
    int n_blocks, blocks_per_xcd, G;
};

// Which (token block, 32-row tile) pairs an interval mask leaves alive: a tile is alive for the blocks of its hull, the
// smallest range of whole token blocks that holds every key some row of the tile sees.  The dQ kernel takes its row tiles,
// groups of LIVE_GROUP row tiles, over the hull of the group, and reads a tile's dS^T inside the tile's own hull only.
// (With whole groups alive or not, 2 x 3000 rows that see the image before them visited 13 % more pairs, since images
// begin inside groups: bwd_kernel 689 us, 599 now, forward and backward 1144 -> 1067)
constexpr int LIVE_GROUP = 8;
constexpr int MAX_RANKED_GROUPS = 1024;    // groups of a launch that are still ranked by length
struct LiveParams {
    const int32_t* kv_len;     // may be null
    const int32_t* kv_start;
    const int32_t* kv_end;
    int32_t* tile_hull;        // out: [B][n_tiles][2] token range of a row tile (multiples of 128), (0, 0) if empty
    int32_t* live_runs;        // out, see BwdParams; of more than four runs those the smallest gaps apart
                               // become one (visiting more is harmless)
    int32_t* order;            // out (may be null): the B * n_groups group indices b * n_groups + grp,
                               // longest hull first (ties in index order)
    int B, Lq, Lkv, row_begin, row_end, n_tiles, n_groups, n_kv_blocks;
    PlanParams plan;           // only where live_in_one
    Divisor by_tiles;          // filled in by launch_bwd_meta, by n_tiles
};
// Whether one launch writes all three, its work-groups taking the hulls they need themselves instead of waiting for a launch of them:
// each reads all intervals of a sample, and one those of all samples, 256 rows in a wave's 0.5 us.
constexpr int MAX_LIVE_TILES = 512;
inline bool live_in_one(const LiveParams& p) { return (int64_t)p.B * p.n_groups * LIVE_GROUP <= MAX_LIVE_TILES; }
// has_hulls: launch_bwd_meta has been given the same (and written tile_hull, or all three)
hipError_t launch_bwd_live(const LiveParams& p, hipStream_t st, bool has_hulls);

// The token blocks of a backward launch that several work-groups share, hence whose dK / dV are summed in the
// fp32 scratch [2][B, Lkv, Hkv, D].  They are listed (b, kv head, block) with the block fastest, the
// sample next; XCD x takes blocks_per_xcd of them and shares all but its first `whole`.
struct SharedBlocks {
    int B, Hkv, Lkv, D, n_kv_blocks, n_blocks, blocks_per_xcd, whole;
};

// Row metadata of the backward in the form its kernel consumes, one 256-byte
// record per (b, h, 32-row tile of the window).
struct MetaParams {
    const float* lse;
    const float* delta;
    float* out;
    int B, Hq, Lq, row_begin, row_end, n_tiles;
    // one launch for `rounds` windows of round_rows rows each (n_tiles: of one of them; the last may have fewer), whose
    // records are round_out floats apart
    int rounds, round_rows;
    int64_t round_out;
    float scale;
    // not null: delta is formed from these and not read
    const uint16_t* o;
    const uint16_t* dout;
    Strides3 os, ds;
    int D, f16;
    float* scratch;            // null, or the fp32 dK / dV scratch whose shared token blocks the same launch zeroes
    SharedBlocks sb;
    // filled in by the launcher: blocks [0, table_blocks) write the tables of `live` (or, not with `tables`, its tile_hull only),
    // those up to meta_end the records (in every window, blockIdx.y), the others zero the scratch
    int table_blocks, tables, meta_end;
    Divisor by_rows, by_Hq;    // by the rows of the window's whole tiles, by q heads
    LiveParams live;
};

// The shared token blocks of the scratch, rounded into dK and dV.
struct CastSharedParams {
    SharedBlocks sb;
    const float* scratch;
    uint16_t* dk;
    uint16_t* dv;
    Strides3 dks, dvs;
    int f16;
};

// The blocks that have been cut: their slices added and rounded into dK and dV.
struct CastSlicesParams {
    const uint32_t* shared;    // of a plan, [8][shared_max][SHARED_ENTRY]; null: an XCD shares all but its first `whole` blocks, `mid` of
    int shared_max;            // them among `splits` and the others among `splits2` work-groups
    int whole, mid, splits, splits2, slices_per_xcd, n_blocks, blocks_per_xcd;
    const float* slices;
    int B, Lkv, D, n_kv_blocks, f16;
    uint16_t* dk;
    uint16_t* dv;
    Strides3 dks, dvs;
};
hipError_t launch_cast_slices(const CastSlicesParams& p, hipStream_t st);

constexpr int SHARE_PARTS = 4;          // work-groups to a block
inline int cast_slices_blocks(const CastSlicesParams& p) { return 8 * p.shared_max * SHARE_PARTS; }

// dQ = (scale dS) K of a window of `rows` rows, from the dS^T workspace.
struct DqParams {
    const uint16_t* ds;        // dS^T tiles [B * Hq][token blocks][row tiles][16 groups of tokens][32 rows][8 tokens]
    int64_t ds_bh;             // elements per (b, h)
    const uint16_t* k;
    uint16_t* dq;              // of the window's first row
    Strides3 ks, dqs;
    int B, Hq, G, rows, row_tiles, Lkv;
    int D;                     // head dimension: 16, 32, 64 or 128
    int f16;                   // element type of dS^T, k and dq
    int stream;                // 1: dS^T is loaded with the streaming hint
    const int32_t* kv_len;     // null or [B]: tokens past it are not contracted
    // Null, or [B][row_tiles][2]: the tokens at which a row tile holds anything, first and one-past-last (multiples of
    // 128; 0, 0: nowhere).  Elsewhere it counts as zeros and is not read.
    const int32_t* tile_range;
    int few;                   // 1: dq_few_kernel, work-groups of DQ_FEW_TILES row tiles (0: of eight)
    // With tile_range and one split, not few: the (sample, group of 8 row tiles) pairs b * groups + group in the order the work-groups
    // are to take them, longest first (null: in index order).
    const int32_t* order;
    // k_splits > 1: as many work-groups per tile of dQ, each contracting split_len tokens (a multiple of 128) into
    // an fp32 slice of its own, part[split * part_split + (b * Hq + h) * D * rows + d * rows + row] (zeros where its range
    // is empty); the caller sums the slices.
    int k_splits, split_len;
    float* part;
    int64_t part_split;
    // filled in by launch_dq
    int total_wg;
    Divisor by_splits, by_tiles_m, by_B, by_Hq, by_G;
    int cast_wg;               // the first so many work-groups (a multiple of 8) do this, which is dK's and dV's
    CastSlicesParams cast;
};
hipError_t launch_dq(const DqParams& p, hipStream_t st, const CastSlicesParams* cast = nullptr);

// One GEMM problem C[M,N] = sum over segments A_s[M,K_s] * B_s[K_s,N].
struct GemmProblem {
    const uint16_t* A[2];
    const uint16_t* Bm[2];
    int64_t lda[2], ldb[2];
    int K[2];
    int nseg;
    uint16_t* C;
    int64_t ldc;
};

// `nprob` problems of one shape.
struct GemmParams {
    GemmProblem prob[2];
    int nprob;
    int M, N;
    int tiles_m, tiles_n, total_wg;   // filled in by launch_gemm for the tile it picks
    // RMS norm over each aligned group of 128 columns of problem 0's C (the k_norm of the K
    // projection), applied to the accumulator before the store: y = bf16(w * bf16(x * r)),
    // r = rsqrt(mean(x^2) + eps), x = the bf16-rounded product.  norm_w: 128 bf16 weights
    // (null: off).  c_raw (optional): x itself, indexed like C.  rstd (optional):
    // r[m * (N / 128) + n / 128].
    const uint16_t* norm_w;
    float norm_eps;
    uint16_t* c_raw;
    float* rstd;
    int f16;                   // element type of A, B, C (and the norm weight): 0 bf16, 1 fp16
    Divisor by_tiles_n, by_tiles_m, by_nprob;      // filled in by launch_gemm: divisors by tiles_n, tiles_m, nprob
};

// p.bias selects the bias variant.  before: null, or parts that the launch folds on its way (wide form only, see fold_rides)
hipError_t launch_fwd(const FwdParams& p, bool masked, hipStream_t st, const FwdFold* before = nullptr);
hipError_t launch_merge(const MergeParams& p, hipStream_t st);
hipError_t launch_preprocess(const PreParams& p, hipStream_t st);
hipError_t launch_bwd(const BwdParams& p, bool masked, hipStream_t st, const CastParams* dq_before = nullptr);
hipError_t plan_cast_t(CastParams& p, int threads);
hipError_t launch_cast(const CastParams& p, hipStream_t st);
hipError_t launch_cast_shared(const CastSharedParams& p, hipStream_t st);
// live: null, or what has its tables, or with many row tiles its hulls, written by the same launch (of one window)
hipError_t launch_bwd_meta(const MetaParams& p, hipStream_t st, const LiveParams* live = nullptr);

// Backward of the 128-wide RMS norm: rows of dy, x [M][heads][128] (row strides ldy, ldx), r [M][heads].
struct NormBwdParams {
    const uint16_t* dy;
    const uint16_t* x;
    const float* rstd;
    const uint16_t* w;
    uint16_t* dx;
    float* dw;        // [128] fp32, added to (null: not wanted)
    int64_t ldy, ldx, lddx;
    int M, heads;
    int f16;
};
hipError_t launch_norm_bwd(const NormBwdParams& p, hipStream_t st);
// a_mcontig: A is stored [K][M] (m contiguous); b_ncontig: B is stored [K][N].
hipError_t launch_gemm(const GemmParams& p, bool a_mcontig, bool b_ncontig, hipStream_t st);

}  // namespace lvx

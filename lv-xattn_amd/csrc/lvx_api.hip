// C-ABI layer: argument validation on the host (nothing is launched when a
// check fails), translation to the internal launch parameters, error strings.
#include "../../include/lvx.h"
#include "lvx_dq_rule.hpp"
#include "lvx_fold.hpp"
#include "lvx_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>

using namespace lvx;

namespace {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_tensor(const lvx_tensor* t) {
    if (!t || !t->ptr) return LVX_ERR_NULL;
    if (!aligned16(t->ptr)) return LVX_ERR_ALIGN;
    if ((t->stride_b % 8) || (t->stride_h % 8) || (t->stride_s % 8)) return LVX_ERR_ALIGN;
    if (t->stride_s <= 0) return LVX_ERR_SHAPE;
    return LVX_OK;
}

int check_shape(const lvx_attn_shape* s) {
    if (!s) return LVX_ERR_NULL;
    if (s->dtype != LVX_BF16 && s->dtype != LVX_F16) return LVX_ERR_DTYPE;
    if (s->D != 128 && s->D != 64 && s->D != 32 && s->D != 16) return LVX_ERR_HEAD_DIM;
    if (s->B <= 0 || s->Hq <= 0 || s->Hkv <= 0 || s->Lq <= 0 || s->Lkv <= 0) return LVX_ERR_SHAPE;
    if (s->Hq % s->Hkv) return LVX_ERR_SHAPE;
    if (!(s->scale > 0.f) || !std::isfinite(s->scale)) return LVX_ERR_SCALE;
    if ((s->kv_start == nullptr) != (s->kv_end == nullptr)) return LVX_ERR_NULL;
    if (s->bias) {
        // rows are read in groups of 4 keys with 16-byte loads: every row must start on a
        // 16-byte boundary and be readable up to Lkv rounded up to 4
        if (reinterpret_cast<uintptr_t>(s->bias) & 15) return LVX_ERR_ALIGN;
        if ((s->bias_stride_r | s->bias_stride_h | s->bias_stride_b) & 3) return LVX_ERR_ALIGN;
        if (s->bias_stride_r < (s->Lkv + 3) / 4 * 4) return LVX_ERR_SHAPE;
    }
    return LVX_OK;
}

int check_rows(const lvx_attn_shape* s, int32_t row_begin, int32_t row_count) {
    if (row_begin < 0 || row_count < 0 || (int64_t)row_begin + row_count > s->Lq) return LVX_ERR_SHAPE;
    return LVX_OK;
}

inline Strides3 st3(const lvx_tensor* t) { return Strides3{t->stride_b, t->stride_h, t->stride_s}; }

inline int gcd(int a, int b) { return b ? gcd(b, a % b) : a; }

constexpr float LOG2E = 1.4426950408889634f;
constexpr int FWD_BN = 64;
constexpr int MAX_SPLITS = 64;

#define LVX_TRY(expr)            \
    do {                         \
        int rc_ = (expr);        \
        if (rc_ != LVX_OK) return rc_; \
    } while (0)

}  // namespace

static void fill_grid(GemmParams& g, int M, int N, int nprob);

// Device memory of lvx_fwd_noalloc: the key-split partials live in this file-scope array
// instead of a caller's workspace.  Every GPU the library runs on holds its own copy at its
// own address until the process ends; the address is asked for once per device.
constexpr size_t NOALLOC_SCRATCH_BYTES = LVX_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex scratch_mutex;
void* scratch_ptr[MAX_DEVICES];      // per device: where that device keeps `scratch`

// The device address of `scratch` on the current device (the array's name is a host-side
// stand-in, not an address a kernel can use).
int scratch_on_current_device(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return static_cast<int>(e);
    if (dev < 0 || dev >= MAX_DEVICES) return LVX_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return static_cast<int>(e);
        if (!ptr) return LVX_ERR_UNSUPPORTED;
        scratch_ptr[dev] = ptr;
    }
    *out = scratch_ptr[dev];
    return LVX_OK;
}
}  // namespace

namespace lvx {
int cu_count() {
    static int cached[MAX_DEVICES];          // 0: not asked yet
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return 256;
    int n = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        __atomic_store_n(&cached[dev], n, __ATOMIC_RELAXED);
    }
    return n;
}
}  // namespace lvx

extern "C" {

int lvx_version(void) { return LVX_VERSION; }

int lvx_max_rounds(void) { return 1 << 18; }        // what fits an int32 above the splits

const char* lvx_strerror(int code) {
    switch (code) {
        case LVX_OK: return "ok";
        case LVX_ERR_NULL: return "a required pointer is NULL";
        case LVX_ERR_ALIGN: return "pointer not 16-byte aligned or stride not a multiple of 8 elements";
        case LVX_ERR_SHAPE: return "bad sizes or row window";
        case LVX_ERR_HEAD_DIM: return "head_dim must be 16, 32, 64 or 128";
        case LVX_ERR_DTYPE: return "dtype must be LVX_BF16 or LVX_F16";
        case LVX_ERR_SCALE: return "scale must be finite and > 0";
        case LVX_ERR_WORKSPACE: return "workspace missing or too small";
        case LVX_ERR_UNSUPPORTED: return "not supported by this build";
        default: break;
    }
    if (code > 0) return hipGetErrorString(static_cast<hipError_t>(code));
    return "unknown lvx error";
}

// The rounds that kv_splits asks for (1: none), taken out of it.
static int fwd_rounds(int32_t& kv_splits) {
    const int rounds = kv_splits > 0 ? kv_splits >> 12 : 0;
    if (rounds > 0) kv_splits &= (1 << 12) - 1;
    return std::max(rounds, 1);
}

static bool parts_ride(const lvx_attn_shape* s, int rows, int kv_splits);

// The room that the parts of one of several blocks of `rows` rows take, a multiple of 16; twice that where they wait for the next block.
static size_t round_parts(const lvx_attn_shape* s, int rows, int32_t kv_splits) {
    return (lvx_fwd_workspace_bytes(s, rows, kv_splits) + 15) / 16 * 16;
}

size_t lvx_fwd_workspace_bytes(const lvx_attn_shape* s, int32_t row_count, int32_t kv_splits) {
    if (const int rounds = fwd_rounds(kv_splits); rounds > 1 && s && row_count > 0) {
        const int rows = (int)(((int64_t)row_count + rounds - 1) / rounds);
        return round_parts(s, rows, kv_splits) * (parts_ride(s, rows, kv_splits) ? 2 : 1);
    }
    const bool f32 = kv_splits > 0 && (kv_splits & LVX_SPLITS_FP32);
    if (f32) kv_splits &= ~LVX_SPLITS_FP32;
    if (!s || kv_splits <= 1 || row_count <= 0) return 0;
    const size_t rows = (size_t)s->B * s->Hq * row_count;
    return (size_t)kv_splits * rows * (s->D * (f32 ? sizeof(float) : sizeof(uint16_t)) + sizeof(float));
}

// Keys per split: whole tiles (pieces) of the form's kernel.
static int fwd_split_len(const lvx_attn_shape* s, FwdForm form, int splits) {
    const int step = form == FWD_FEW ? 32 : FWD_BN;
    return ((s->Lkv + splits - 1) / splits + step - 1) / step * step;
}

// What a forward launch over `rows` text rows in this form with this many key splits takes, in us; the
// constants are fits to launches of 1 .. 4096 rows against 600 .. 76848 keys:
//   few  : 5 us, and per key of a work-group's range 8 ns (4.2 with heads of 64, 3 below) together with
//          the time HBM takes for K and V (the root of the sum of squares: the two overlap in part).  One row x 32 heads x 6404 keys: 46 us whole, 12.5 in 16 - 32 parts;
//          4 rows x 76848 keys in 32 parts: 61 us, 5.2 TB/s
//   wide : 11 us per round of work-groups (fitted before their way in and out got 2 us shorter; with 9 the ranges of 12 in
//          504 launches of 1 to 4096 rows would differ), and per 64-key tile 1.1 us on an idle chip, 1.5 on a full one
//          (0.9 and 1.05 with heads of 64).  256 rows x 6404 keys: 138 us whole, 39 in 8 parts
//   plain: the same with 1.8 us per tile and two work-groups per CU
// with a dense bias and heads of 128 / 64 (launches of 1 .. 2000 rows against 400 .. 13000 keys, ranges of 1 to 64):
//   wide : 7 us per round and per tile 1.65 us on an idle chip, 2.1 on a full one (6 us, 1.45, 1.55)
//   plain: 4 us and 2.15, or 2.8 once CUs have two work-groups (3.5 us, 1.95 and 2.35)
// plus, with splits, 4 us for the launch that folds the parts and their bytes at 4 TB/s, what fp32 adds to them at 9.  With a dense bias and
// heads of 128 and 64 each part takes the fold 0.054 us besides (in the other prices the 11 us of a round stand for it): of 647 such
// launches, ranges that are dearer by over 3 % than those of the plain form at its earlier price are chosen for 6, without it for 19,
// by up to 18 % (142 rows x 3 heads x 3391 keys: 27 ranges 14.5 us, 53 18.3).
struct FwdPrice {
    double tile_us, load_us, round_us;      // per key tile on an idle chip, what a full one adds, per round of work-groups
    bool shared;                            // it is two work-groups on a CU that add it, however many there are
    double part_us;                         // per part, in the fold
};
constexpr FwdPrice PLAIN_PRICE{0.8, 1.0, 11.0, false, 0.0};
static FwdPrice fwd_price(const lvx_attn_shape* s, FwdForm form) {
    const bool wide = form == FWD_WIDE;
    if (s->bias && s->D == 128) return wide ? FwdPrice{1.65, 0.45, 7.0, false, 0.054} : FwdPrice{2.15, 0.65, 4.0, true, 0.054};
    if (s->bias && s->D == 64) return wide ? FwdPrice{1.45, 0.1, 6.0, false, 0.054} : FwdPrice{1.95, 0.4, 3.5, true, 0.054};
    if (!wide) return PLAIN_PRICE;
    return s->D == 128 ? FwdPrice{1.1, 0.4, 11.0, false, 0.0} : FwdPrice{0.9, 0.15, 11.0, false, 0.0};
}

static double fwd_cost(const lvx_attn_shape* s, int rows, FwdForm form, int splits, bool parts_f32, int n_cu, const FwdPrice& price) {
    const int G = s->Hq / s->Hkv, hg = gcd(G, 4), rs = 4 / hg;
    const int64_t split_len = fwd_split_len(s, form, splits);
    const int64_t n = (s->Lkv + split_len - 1) / split_len;
    const double fold_us = (4 * s->D + 8) / 4e6 + (parts_f32 ? 4 * s->D / 9e6 : 0.0);       // per row, head and part
    double t = n > 1 ? 4.0 + n * price.part_us + (double)n * s->B * s->Hq * rows * fold_us : 0.0;
    if (form == FWD_FEW) {
        const int64_t wgs = (int64_t)s->B * s->Hkv * (((int64_t)rows * G + 31) / 32) * n;
        const int64_t slots = s->D == 128 ? n_cu : 2 * n_cu;
        const double key_us = s->D == 128 ? 8e-3 : s->D == 64 ? 4.2e-3 : 3e-3;
        const double hbm_us = (double)s->B * s->Hkv * s->Lkv * s->D * 4 / 5.2e6;
        return t + 5.0 + std::hypot((double)((wgs + slots - 1) / slots) * (split_len * key_us + 3.0) - 3.0, hbm_us);
    }
    const int wg_rows = (form == FWD_WIDE ? 64 : 32) * rs;
    const int64_t wgs = (int64_t)s->B * (s->Hq / hg) * ((rows + wg_rows - 1) / wg_rows) * n;
    const int64_t slots = form == FWD_WIDE ? n_cu : 2 * n_cu;
    const double tile_us = price.tile_us + price.load_us * (price.shared ? (wgs > n_cu ? 1.0 : 0.0) : std::min(1.0, (double)wgs / slots));
    return t + (double)((wgs + slots - 1) / slots) * (split_len / FWD_BN * tile_us + price.round_us);
}
static double fwd_cost(const lvx_attn_shape* s, int rows, FwdForm form, int splits, bool parts_f32, int n_cu) {
    return fwd_cost(s, rows, form, splits, parts_f32, n_cu, fwd_price(s, form));
}

// A second, closer fit, for launches without a dense bias: what the forms take by now, among them the fold inside a launch for few rows, K
// and V from memory in every form.  900 random launches (1 .. 2500 rows against 300 .. 40000 keys, all head dimensions, K and V not in the
// caches): the ranges and the form it finds cheapest are 1.7 % from the best on average, those of the one above 3.4.  (A work-group for few rows that
// shares its CU takes longer per key, with heads of 64 by half; and a load of the fold inside a launch holds 2048 / D parts.  With one price for both, and
// for parts of any size, short launches and small heads were cut where that costs: 155 rows x 3 x 16 heads of 64 x 2652 keys 17.5 us whole,
// 19.8 in two parts, 3 x 2 x 2 of 32 x 12498 7.5 in 56, 8.6 in 23.)
static double fwd_cost2(const lvx_attn_shape* s, int rows, FwdForm form, int splits, bool parts_f32, int n_cu) {
    struct Fit { double key_us, key2_us, tile_us, load_us, round_us; };     // per key of a work-group that has its CU to itself, that shares it
    const Fit f = s->D == 128 ? Fit{7.7e-3, 7.7e-3, 1.2, 0.26, 4.5} : s->D == 64 ? Fit{4.4e-3, 6.9e-3, 1.1, 0.0, 3.4}
                : s->D == 32 ? Fit{3.8e-3, 5.3e-3, 1.2, 0.2, 1.6} : Fit{3.7e-3, 4.9e-3, 1.1, 0.0, 1.7};
    const int G = s->Hq / s->Hkv, hg = gcd(G, 4);
    const int64_t split_len = fwd_split_len(s, form, splits), n = (s->Lkv + split_len - 1) / split_len;
    const auto both = [](double x, double y) { return std::sqrt(x * x + y * y); };      // (hypot takes three times as long, for ranges that are not ours)
    const double kv_mb = (double)s->B * s->Hkv * s->Lkv * s->D * 4e-6;
    double t = 0.0;
    if (n > 1 && form == FWD_FEW && fold_inside((int)n, (int64_t)rows * G)) t = (s->D == 128 ? 2.4 : 1.5) + 0.054 * n * s->D / 128;
    else if (n > 1) t = 3.4 + 0.054 * n + (double)n * s->B * s->Hq * rows * ((4 * s->D + 8) / 6.9e6 + (parts_f32 ? 4 * s->D / 7.1e6 : 0.0));
    const int64_t slots = form == FWD_WIDE || (form == FWD_FEW && s->D == 128) ? n_cu : 2 * n_cu;
    if (form == FWD_FEW) {
        const int64_t wgs = (int64_t)s->B * s->Hkv * (((int64_t)rows * G + 31) / 32) * n;
        return t + 2.9 + both((double)((wgs + slots - 1) / slots) * (split_len * (wgs <= n_cu ? f.key_us : f.key2_us) + 3.2) - 3.2, kv_mb / 6.8);
    }
    const int wg_rows = (form == FWD_WIDE ? 64 : 32) * (4 / hg);
    const int64_t wgs = (int64_t)s->B * (s->Hq / hg) * (((int64_t)rows + wg_rows - 1) / wg_rows) * n;
    const double tile_us = f.tile_us + f.load_us * std::min(1.0, (double)wgs / slots);
    return t + both((double)((wgs + slots - 1) / slots) * (split_len / FWD_BN * tile_us + f.round_us), kv_mb / 8.2);
}

// The form for few rows is for up to 256 (row, head) columns per kv head: it reads K and V from L2 once
// per 32 of them, and with more the other forms only lose where they are cut into too few splits.
constexpr int64_t FEW_MAX_COLS = 256;
static bool fwd_few_ok(const lvx_attn_shape* s, int rows) {
    return !s->bias && (int64_t)rows * (s->Hq / s->Hkv) <= FEW_MAX_COLS;
}

// The forms that a shape's launches may have: heads of 128 and 64 take the wide form or, where reading K and V is the
// larger part of the work, the form for few rows; the plain one was slower at every size measured
// (4096 rows x 6404 keys: 429 us against 354; 300 rows x 2 samples: 92 against 88) and is not built for them without a dense
// bias.  With one the wide form wins where there are enough rows for its work-groups of 64 per wave, the plain one where
// there are few, its work-groups being two to a CU and its way in and out shorter.  us with the best number of ranges, plain / wide:
// 1024 rows x 16 heads x 4096 keys 61.6 / 53.7 (heads of 64 50.1 / 40.1), 1024 x 32 x 6404 152 / 130, 3 x 2000 x 16 x 2500 213 / 175,
// 2 x 700 x 32 x 800 of 64 43.9 / 27.2, 256 x 16 x 4096 30.0 / 27.2; 1 x 16 x 4096 14.0 / 18.2, 33 x 16 x 13000 31.9 / 36.6, 300 x 8 x
// 3000 20.2 / 22.0.  (A row of a bias in bytes is a factor of 24 bits in the wide form.)
static bool fwd_form_ok(const lvx_attn_shape* s, int rows, FwdForm form) {
    const bool heads = s->D == 128 || s->D == 64;
    if (form == FWD_FEW) return fwd_few_ok(s, rows);
    if (form == FWD_PLAIN) return !heads || s->bias;
    return heads && (!s->bias || s->bias_stride_r < (1 << 22));
}
constexpr FwdForm FWD_FORMS[] = {FWD_PLAIN, FWD_WIDE, FWD_FEW};

// What the closer fit has to promise before a launch takes another form or other ranges than the first one says.  Of 12000 random launches 592
// then do, 450 of them faster by over 3 % (few rows of many keys by up to 32), 12 slower by up to 9.  (Of 900 others 30 and 2;
// at 1.05 107 and 12, without it 184 and 30 by up to 22.)
constexpr double CLOSER_FIT = 1.12;

// The form of the forward kernel for a window of `rows` rows whose keys are cut into `splits` ranges.
static FwdForm fwd_form(const lvx_attn_shape* s, int rows, int splits, bool parts_f32) {
    const char* const e = getenv("LVX_FWD_WIDE");
    FwdForm ok[3];
    int n = 0;
    for (const FwdForm form : FWD_FORMS) {
        if (!fwd_form_ok(s, rows, form)) continue;
        if (e && form == (atoi(e) == 2 ? FWD_FEW : FWD_WIDE)) return form;
        if (e && form == FWD_FEW) continue;
        ok[n++] = form;
    }
    if (n == 1) return ok[0];
    double first[3], closer[3];
    int a = 0, b = 0;                   // cheapest by either fit
    const int n_cu = cu_count();
    for (int i = 0; i < n; ++i) {
        first[i] = fwd_cost(s, rows, ok[i], splits, parts_f32, n_cu);
        closer[i] = s->bias ? 0.0 : fwd_cost2(s, rows, ok[i], splits, parts_f32, n_cu);
        if (first[i] < first[a] || (ok[i] == FWD_FEW && first[i] == first[a])) a = i;
        if (closer[i] < closer[b]) b = i;
    }
    return ok[closer[a] <= CLOSER_FIT * closer[b] ? a : b];
}

// Whether the parts of a launch whose splits are chosen here wait for the fold in fp32.  In 16 bits they are a
// rounding that a launch of one range does not have: relative error against 64 bits 2.83e-3 instead of 2.32e-3
// (bf16, N(0, 1) inputs), whatever the number of parts.  The form for few rows has little O: fp32 does not show in
// a decoded token (one row x 6404 keys 10.2 us in 16 bits, 10.3 in fp32) and costs 4 % at 145 (row, head) columns per
// kv head (four rounds of 145 rows, 3 x 8 heads of 32, 8149 keys: 74.9 us, 77.9).  In the others fp32 costs 2 - 7 % of the launch, and cutting
// either is what fills the chip - fewer than two work-groups of 32-row waves per CU, ranges of 512 keys and
// more: 256 rows x 6404 keys 137 us whole, 37.4 in 8 parts, 40.1 with those in fp32 - where they stay in 16
// bits, or it only evens out the last round of work-groups (2100 rows x 6404 keys 310 us whole, 263 in 2 parts, 270
// with those in fp32) or cuts a short range shorter: there the result keeps the precision of the whole launch.
static bool fwd_parts_f32(const lvx_attn_shape* s, int rows, FwdForm form) {
    if (form == FWD_FEW) return true;
    const int hg = gcd(s->Hq / s->Hkv, 4), wg_rows = 32 * (4 / hg);
    const int64_t wgs = (int64_t)s->B * (s->Hq / hg) * (((int64_t)rows + wg_rows - 1) / wg_rows);
    return wgs >= 2 * cu_count() || s->Lkv < 1024;
}

int lvx_fwd_auto_splits(const lvx_attn_shape* s, int32_t row_count) {
    if (check_shape(s) != LVX_OK || row_count <= 0) return 1;
    const int n_cu = cu_count();
    // The number of ranges for less than best_cost (0: for any), or 0.
    const auto cheapest = [&](FwdForm form, bool f32, const FwdPrice& price, double& best_cost) {
        int best = 0;
        for (int n = 1; n <= MAX_SPLITS && (n == 1 || s->Lkv / n >= 32); ++n) {
            const double c = fwd_cost(s, row_count, form, n, f32, n_cu, price);
            if (best_cost == 0.0 || c < best_cost) { best = n; best_cost = c; }
        }
        return best;
    };
    // With a dense bias, parts are in 16 bits only where the plain form at the price it has without one would be cut: a launch that only the
    // prices with a bias cut keeps the precision of the whole one, in either form.
    double plain_cost = 0.0;
    const bool only_here = s->bias && cheapest(FWD_PLAIN, fwd_parts_f32(s, row_count, FWD_PLAIN), PLAIN_PRICE, plain_cost) == 1;
    int best = 1;
    double best_cost = 0.0;
    for (const FwdForm form : FWD_FORMS) {
        if (!fwd_form_ok(s, row_count, form)) continue;
        const bool f32 = only_here || fwd_parts_f32(s, row_count, form);
        if (const int n = cheapest(form, f32, fwd_price(s, form), best_cost)) best = n > 1 && f32 ? n | LVX_SPLITS_FP32 : n;
    }
    if (s->bias) return best;
    // Parts are in 16 bits only where those of the first fit are: not where it leaves the launch whole, nor where it takes the form for few
    // rows, in whichever form they then come about.
    const bool f32 = best == 1 || (best & LVX_SPLITS_FP32);
    const auto parts = [&](int n, FwdForm form) { return n > 1 && (f32 || form == FWD_FEW) ? n | LVX_SPLITS_FP32 : n; };
    int best2 = 1;
    double best2_cost = 0.0;
    for (const FwdForm form : FWD_FORMS)
        for (int n = 1; fwd_form_ok(s, row_count, form) && n <= MAX_SPLITS && (n == 1 || s->Lkv / n >= 32); ++n) {
            const double c = fwd_cost2(s, row_count, form, n, parts(n, form) != n, n_cu);
            if (best2_cost == 0.0 || c < best2_cost) { best2 = parts(n, form); best2_cost = c; }
        }
    const int n = best & ~LVX_SPLITS_FP32;
    const FwdForm form = fwd_form(s, row_count, n, best != n);
    if (fwd_cost2(s, row_count, form, n, best != n, n_cu) > CLOSER_FIT * best2_cost) return best2;
    return form == FWD_FEW ? parts(n, form) : best;
}

struct FwdGrid {
    int row_tiles, head_groups;
    int64_t wgs;
};

static FwdGrid fwd_grid(const lvx_attn_shape* s, int rows, FwdForm form, int nsplit) {
    const int G = s->Hq / s->Hkv, hg = gcd(G, 4);
    FwdGrid g;
    if (form == FWD_FEW) {
        g.row_tiles = (rows * G + 31) / 32;               // tiles of 32 (row, head of the group) columns
        g.head_groups = s->Hkv;
    } else {
        const int wg_rows = (form == FWD_WIDE ? 64 : 32) * (4 / hg);
        g.row_tiles = (rows + wg_rows - 1) / wg_rows;
        g.head_groups = s->Hq / hg;
    }
    g.wgs = (int64_t)s->B * g.head_groups * nsplit * g.row_tiles;
    return g;
}

// Whether blocks of `rows` rows, one after the other, leave their parts to the launch of the next.  A shape that does not say how
// many keys and kv heads there are may.
static bool parts_ride(const lvx_attn_shape* s, int rows, int kv_splits) {
    if (kv_splits <= 1 || kv_splits > MAX_SPLITS || s->bias || (s->D != 128 && s->D != 64)) return false;     // (LVX_SPLITS_FP32 among them)
    if (s->B <= 0 || s->Hq <= 0) return false;      // (nothing has been checked yet where only the room is asked for)
    if (s->Hkv <= 0 || s->Hq % s->Hkv || s->Lkv <= 0) return true;
    if (fwd_form(s, rows, kv_splits, false) != FWD_WIDE) return false;
    const int split_len = fwd_split_len(s, FWD_WIDE, kv_splits), nsplit = (s->Lkv + split_len - 1) / split_len;
    return fold_rides(nsplit, (int64_t)s->B * s->Hq * rows, s->D / 8, fwd_grid(s, rows, FWD_WIDE, nsplit).wgs, cu_count());
}

// The fold of one block's 16-bit parts as a launch of its own.
static int fold_parts(const lvx_attn_shape* s, const FwdFold& f, hipStream_t st) {
    MergeParams m{};
    m.f16 = s->dtype == LVX_F16;
    m.D = s->D;
    m.o_acc = f.o - (int64_t)f.row_begin * f.os.s;
    m.l_acc = f.l;
    m.oa = f.os;
    m.o_part = f.part - (int64_t)f.row_begin * s->D;
    m.l_part = f.l_part - f.row_begin;
    m.op = Strides3{(int64_t)s->Hq * f.rows * s->D, (int64_t)f.rows * s->D, s->D};
    m.l_part_stride = (int64_t)s->B * s->Hq * f.rows;
    m.o_part_stride = m.l_part_stride * s->D;
    m.l_acc_bh = s->Lq;
    m.l_part_bh = f.rows;
    m.nparts = f.nparts;
    if (f.acc) {
        m.use_acc = 1;
        m.o_in = f.acc - (int64_t)f.row_begin * f.as.s;
        m.l_in = f.l_acc;
        m.oi = f.as;
        m.l_in_bh = s->Lq;
    }
    m.B = s->B; m.Hq = s->Hq; m.Lq = s->Lq;
    m.row_begin = f.row_begin; m.row_end = f.row_begin + f.rows;
    return static_cast<int>(launch_merge(m, st));
}

// Whether the memory that o spans has any of q, k and v in it, which a launch that folds its own parts may not yet have read when o is first
// written to.
static bool overlap(const lvx_attn_shape* s, const lvx_tensor* o, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v) {
    const auto end = [&](const lvx_tensor* t, int heads, int rows, int sign) {      // the last element, or before the first (strides may be negative)
        int64_t at = 0;
        const int64_t steps[3] = {(s->B - 1) * t->stride_b, (heads - 1) * t->stride_h, (rows - 1) * t->stride_s};
        for (const int64_t x : steps) at += sign * x > 0 ? x : 0;
        return static_cast<const uint16_t*>(t->ptr) + at + (sign > 0 ? s->D : 0);
    };
    const auto meets = [&](const lvx_tensor* t, int heads, int rows) {
        return end(o, s->Hq, s->Lq, -1) < end(t, heads, rows, 1) && end(t, heads, rows, -1) < end(o, s->Hq, s->Lq, 1);
    };
    return meets(q, s->Hq, s->Lq) || meets(k, s->Hkv, s->Lkv) || meets(v, s->Hkv, s->Lkv);
}

// lvx_fwd, and lvx_fwd_acc when (o_in, l_in) is given: the result is then merged with that
// incoming accumulator before it is written to (o, lse).
static int fwd_impl(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v,
                    const lvx_tensor* o, float* lse, int32_t row_begin, int32_t row_count, int32_t kv_splits,
                    void* workspace, size_t workspace_bytes, void* stream, const lvx_tensor* o_in, const float* l_in,
                    FwdFold* before = nullptr) {
    LVX_TRY(check_shape(s));
    LVX_TRY(check_tensor(q));
    LVX_TRY(check_tensor(k));
    LVX_TRY(check_tensor(v));
    LVX_TRY(check_tensor(o));
    if (!lse) return LVX_ERR_NULL;
    LVX_TRY(check_rows(s, row_begin, row_count));
    if (const int rounds = fwd_rounds(kv_splits); rounds > 1) {
        // one launch per block; where the parts of a block wait for the launch that folds them, `parts` carries them there
        const int rows = (row_count + rounds - 1) / rounds;
        const bool ride = row_count > 0 && parts_ride(s, rows, kv_splits);
        const size_t each = round_parts(s, rows, kv_splits);
        if (each && (!workspace || workspace_bytes < each * (ride ? 2 : 1))) return LVX_ERR_WORKSPACE;
        if (each && !aligned16(workspace)) return LVX_ERR_ALIGN;
        FwdFold parts{};
        char* ws = each ? static_cast<char*>(workspace) : nullptr;
        for (int r = 0; r * rows < row_count; ++r) {
            // the other half only while parts wait in the one before: blocks that fold at once keep theirs in the caches
            if (parts.part) ws = ws == workspace ? ws + each : static_cast<char*>(workspace);
            LVX_TRY(fwd_impl(s, q, k, v, o, lse, row_begin + r * rows, std::min(rows, row_count - r * rows), kv_splits, ws, each,
                             stream, o_in, l_in, ride ? &parts : nullptr));
        }
        return parts.part ? fold_parts(s, parts, static_cast<hipStream_t>(stream)) : LVX_OK;
    }
    const int f32 = kv_splits > 0 ? kv_splits & LVX_SPLITS_FP32 : 0;
    kv_splits -= f32;
    if (kv_splits < 1 || kv_splits > MAX_SPLITS) return LVX_ERR_SHAPE;
    if (row_count == 0) return LVX_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);

    FwdParams p{};
    p.f16 = s->dtype == LVX_F16;
    p.D = s->D;
    p.q = static_cast<const uint16_t*>(q->ptr);
    p.k = static_cast<const uint16_t*>(k->ptr);
    p.v = static_cast<const uint16_t*>(v->ptr);
    p.qs = st3(q); p.ks = st3(k); p.vs = st3(v);
    p.kv_len = s->kv_len; p.kv_start = s->kv_start; p.kv_end = s->kv_end;
    p.bias = s->bias; p.bias_b = s->bias_stride_b; p.bias_h = s->bias_stride_h; p.bias_r = s->bias_stride_r;
    p.B = s->B; p.Hq = s->Hq; p.Hkv = s->Hkv; p.Lq = s->Lq; p.Lkv = s->Lkv;
    p.G = s->Hq / s->Hkv;
    p.HG = gcd(p.G, 4);
    p.RS = 4 / p.HG;
    p.row_begin = row_begin; p.row_end = row_begin + row_count;
    const FwdForm form = fwd_form(s, row_count, kv_splits, f32 != 0);
    p.form = form;
    p.scale = s->scale; p.scale_log2e = s->scale * LOG2E;

    int nsplit = kv_splits;
    const int split_len = fwd_split_len(s, form, nsplit);
    nsplit = (s->Lkv + split_len - 1) / split_len;
    p.nsplit = nsplit;
    p.split_len = split_len;
    const FwdGrid grid = fwd_grid(s, row_count, form, nsplit);
    p.n_row_tiles = grid.row_tiles;
    p.n_head_groups = grid.head_groups;
    p.total_wg = (int)grid.wgs;

    // (a last block of fewer rows may be computed in another form, or have too few work-groups for what the one before has left)
    const auto rides = [&](int nparts, int rows) {
        return form == FWD_WIDE && fold_rides(nparts, (int64_t)s->B * s->Hq * rows, s->D / 8, grid.wgs, cu_count());
    };
    const FwdFold* along = before && before->part ? before : nullptr;       // what this block's launch folds on its way
    if (along && !rides(along->nparts, along->rows)) {
        LVX_TRY(fold_parts(s, *along, st));
        along = nullptr;
    }
    if (nsplit == 1) {
        p.o = static_cast<uint16_t*>(o->ptr);
        p.os = st3(o);
        p.lse = lse;
        p.lse_bh_stride = s->Lq;
        const hipError_t e1 = launch_fwd(p, s->kv_start != nullptr, st, along);
        if (before) before->part = nullptr;
        if (e1 != hipSuccess || !o_in) return static_cast<int>(e1);
        // one partial, written straight to (o, lse): fold the incoming accumulator into it (the
        // merge is symmetric, so which side is "the accumulator" does not matter)
        MergeParams m{};
        m.f16 = s->dtype == LVX_F16;
        m.D = s->D;
        m.o_acc = static_cast<uint16_t*>(o->ptr);
        m.l_acc = lse;
        m.o_part = static_cast<const uint16_t*>(o_in->ptr);
        m.l_part = l_in;
        m.oa = st3(o);
        m.op = st3(o_in);
        m.l_acc_bh = s->Lq;
        m.l_part_bh = s->Lq;
        m.nparts = 1;
        m.use_acc = 1;
        m.B = s->B; m.Hq = s->Hq; m.Lq = s->Lq;
        m.row_begin = row_begin; m.row_end = row_begin + row_count;
        return static_cast<int>(launch_merge(m, st));
    }

    // key splits: partials [split][B*Hq][row_count][D] + LSE [split][B*Hq][row_count]
    const size_t need = lvx_fwd_workspace_bytes(s, row_count, nsplit | f32);
    if (!workspace || workspace_bytes < need) return LVX_ERR_WORKSPACE;
    if (!aligned16(workspace)) return LVX_ERR_ALIGN;
    const int64_t rows = (int64_t)s->B * s->Hq * row_count;
    uint16_t* o_ws = static_cast<uint16_t*>(workspace);
    const int words = f32 ? 2 : 1;       // of 16 bits per element of a part
    float* l_ws = reinterpret_cast<float*>(o_ws + (int64_t)nsplit * rows * s->D * words);
    if (form == FWD_FEW && f32 && !o_in && fold_inside(nsplit, (int64_t)row_count * p.G) && !overlap(s, o, q, k, v)) {
        p.o = static_cast<uint16_t*>(o->ptr);
        p.os = st3(o);
        p.lse = lse;
        p.lse_bh_stride = s->Lq;
        p.part = reinterpret_cast<float*>(o_ws);
        p.l_part = l_ws;
        return static_cast<int>(launch_fwd(p, s->kv_start != nullptr, st));
    }
    // the kernel indexes partials by absolute row: bias the bases by -row_begin
    p.o = o_ws - (int64_t)row_begin * s->D * words;
    p.o_f32 = f32 != 0;
    p.os = Strides3{(int64_t)s->Hq * row_count * s->D, (int64_t)row_count * s->D, s->D};
    p.o_split_stride = rows * s->D;
    p.lse = l_ws - row_begin;
    p.lse_bh_stride = row_count;
    p.lse_split_stride = rows;
    hipError_t e = launch_fwd(p, s->kv_start != nullptr, st, along);
    if (before) before->part = nullptr;
    if (e != hipSuccess) return static_cast<int>(e);
    if (before && rides(nsplit, row_count)) {
        *before = FwdFold{o_ws, l_ws, static_cast<uint16_t*>(o->ptr) + (int64_t)row_begin * o->stride_s, lse,
                          o_in ? static_cast<const uint16_t*>(o_in->ptr) + (int64_t)row_begin * o_in->stride_s : nullptr, l_in,
                          st3(o), o_in ? st3(o_in) : Strides3{}, nsplit, row_count, row_begin};
        return LVX_OK;
    }

    MergeParams m{};
    m.f16 = s->dtype == LVX_F16;
    m.D = s->D;
    m.o_acc = static_cast<uint16_t*>(o->ptr);
    m.l_acc = lse;
    m.o_part = p.o;
    m.l_part = p.lse;
    m.oa = st3(o);
    m.op = p.os;
    m.o_part_stride = p.o_split_stride;
    m.l_part_stride = p.lse_split_stride;
    m.l_acc_bh = s->Lq;
    m.l_part_bh = row_count;
    m.nparts = nsplit;
    m.part_f32 = p.o_f32;
    m.use_acc = 0;
    if (o_in) {      // the partials and the incoming accumulator in one launch
        m.use_acc = 1;
        m.o_in = static_cast<const uint16_t*>(o_in->ptr);
        m.l_in = l_in;
        m.oi = st3(o_in);
        m.l_in_bh = s->Lq;
    }
    m.B = s->B; m.Hq = s->Hq; m.Lq = s->Lq;
    m.row_begin = row_begin; m.row_end = row_begin + row_count;
    return static_cast<int>(launch_merge(m, st));
}

int lvx_fwd(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v,
            const lvx_tensor* o, float* lse, int32_t row_begin, int32_t row_count, int32_t kv_splits,
            void* workspace, size_t workspace_bytes, void* stream) {
    return fwd_impl(s, q, k, v, o, lse, row_begin, row_count, kv_splits, workspace, workspace_bytes, stream,
                    nullptr, nullptr);
}

int lvx_fwd_acc(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v,
                const lvx_tensor* o_in, const float* l_in, const lvx_tensor* o, float* lse, int32_t row_begin,
                int32_t row_count, int32_t kv_splits, void* workspace, size_t workspace_bytes, void* stream) {
    if (!o_in) return LVX_ERR_NULL;
    LVX_TRY(check_tensor(o_in));
    if (!l_in) return LVX_ERR_NULL;
    // the result is formed out of place: the kernel writes (o, lse) of the window before the merge
    // reads (o_in, l_in), so the row windows of the two may not share memory
    if (o && o_in->ptr == o->ptr) return LVX_ERR_SHAPE;
    if (l_in == lse) return LVX_ERR_SHAPE;
    if (o && o->ptr && s && row_count > 0 && s->B > 0 && s->Hq > 0) {
        auto span = [&](const lvx_tensor* t, const char*& lo, const char*& hi) {
            const int64_t last = (int64_t)(s->B - 1) * t->stride_b + (int64_t)(s->Hq - 1) * t->stride_h +
                                 (int64_t)(row_begin + row_count - 1) * t->stride_s + s->D;
            lo = static_cast<const char*>(t->ptr) + (int64_t)row_begin * t->stride_s * 2;
            hi = static_cast<const char*>(t->ptr) + last * 2;
        };
        const char *alo, *ahi, *blo, *bhi;
        span(o, alo, ahi);
        span(o_in, blo, bhi);
        if (alo < bhi && blo < ahi) return LVX_ERR_SHAPE;
    }
    if (lse && l_in && s && row_count > 0) {
        const int64_t rows = (int64_t)s->B * s->Hq * s->Lq;
        if (l_in < lse + rows && lse < l_in + rows) return LVX_ERR_SHAPE;
    }
    return fwd_impl(s, q, k, v, o, lse, row_begin, row_count, kv_splits, workspace, workspace_bytes, stream,
                    o_in, l_in);
}

size_t lvx_noalloc_scratch_bytes(void) { return NOALLOC_SCRATCH_BYTES; }

int lvx_fwd_noalloc(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v,
                    const lvx_tensor* o, float* lse, int32_t row_begin, int32_t row_count, int32_t kv_splits,
                    void* stream) {
    // argument errors first, as lvx_fwd reports them
    LVX_TRY(check_shape(s));
    if (kv_splits < 1 || (kv_splits & ~LVX_SPLITS_FP32) < 1 || (kv_splits & ~LVX_SPLITS_FP32) > MAX_SPLITS) return LVX_ERR_SHAPE;
    if (row_count > 0 && lvx_fwd_workspace_bytes(s, row_count, kv_splits) > NOALLOC_SCRATCH_BYTES)
        return LVX_ERR_WORKSPACE;     // the partials of this call do not fit the library's own array
    void* ws = nullptr;
    LVX_TRY(scratch_on_current_device(&ws));
    return lvx_fwd(s, q, k, v, o, lse, row_begin, row_count, kv_splits, ws, NOALLOC_SCRATCH_BYTES, stream);
}

int lvx_merge(const lvx_attn_shape* s, const lvx_tensor* o_acc, float* l_acc, const lvx_tensor* o_part,
              const float* l_part, int32_t row_begin, int32_t row_count, void* stream) {
    LVX_TRY(check_shape(s));
    LVX_TRY(check_tensor(o_acc));
    LVX_TRY(check_tensor(o_part));
    if (!l_acc || !l_part) return LVX_ERR_NULL;
    LVX_TRY(check_rows(s, row_begin, row_count));
    MergeParams m{};
    m.f16 = s->dtype == LVX_F16;
    m.D = s->D;
    m.o_acc = static_cast<uint16_t*>(o_acc->ptr);
    m.l_acc = l_acc;
    m.o_part = static_cast<const uint16_t*>(o_part->ptr);
    m.l_part = l_part;
    m.oa = st3(o_acc);
    m.op = st3(o_part);
    m.l_acc_bh = s->Lq;
    m.l_part_bh = s->Lq;
    m.nparts = 1;
    m.use_acc = 1;
    m.B = s->B; m.Hq = s->Hq; m.Lq = s->Lq;
    m.row_begin = row_begin; m.row_end = row_begin + row_count;
    return static_cast<int>(launch_merge(m, static_cast<hipStream_t>(stream)));
}

int lvx_bias_hull(const lvx_attn_shape* s, int32_t* kv_start, int32_t* kv_end, void* stream) {
    LVX_TRY(check_shape(s));
    if (!s->bias || !kv_start || !kv_end) return LVX_ERR_NULL;
    BiasHullParams p{};
    p.bias = s->bias; p.bias_b = s->bias_stride_b; p.bias_h = s->bias_stride_h; p.bias_r = s->bias_stride_r;
    p.kv_start = kv_start; p.kv_end = kv_end;
    p.B = s->B; p.heads = s->bias_stride_h ? s->Hq : 1; p.Lq = s->Lq; p.Lkv = s->Lkv;
    return static_cast<int>(launch_bias_hull(p, static_cast<hipStream_t>(stream)));
}

int lvx_bias_is_interval(const lvx_attn_shape* s, const int32_t* kv_start, const int32_t* kv_end, int32_t* not_interval,
                         void* stream) {
    LVX_TRY(check_shape(s));
    if (!s->bias || !kv_start || !kv_end || !not_interval) return LVX_ERR_NULL;
    BiasHullParams p{};
    p.bias = s->bias; p.bias_b = s->bias_stride_b; p.bias_h = s->bias_stride_h; p.bias_r = s->bias_stride_r;
    p.kv_start = const_cast<int32_t*>(kv_start); p.kv_end = const_cast<int32_t*>(kv_end);
    p.B = s->B; p.heads = s->bias_stride_h ? s->Hq : 1; p.Lq = s->Lq; p.Lkv = s->Lkv;
    p.flag = not_interval;
    return static_cast<int>(launch_bias_interval(p, static_cast<hipStream_t>(stream)));
}

int lvx_mask_intervals(const void* mask, int32_t type, int64_t stride_b, int64_t stride_r, int32_t B, int32_t Lq,
                       int32_t Lkv, int32_t* kv_start, int32_t* kv_end, void* stream) {
    if (!mask || !kv_start || !kv_end) return LVX_ERR_NULL;
    if (type != LVX_BF16 && type != LVX_F16 && type != 0) return LVX_ERR_DTYPE;
    if (reinterpret_cast<uintptr_t>(mask) & (type ? 1 : 3)) return LVX_ERR_ALIGN;
    if (B <= 0 || Lq <= 0 || Lkv <= 0 || (int64_t)B * Lq > INT32_MAX || stride_b < 0 || stride_r < 0) return LVX_ERR_SHAPE;
    const MaskIntervalParams p{mask, stride_b, stride_r, type, kv_start, kv_end, B, Lq, Lkv};
    return static_cast<int>(launch_mask_intervals(p, static_cast<hipStream_t>(stream)));
}

int lvx_bwd_preprocess(const lvx_attn_shape* s, const lvx_tensor* o, const lvx_tensor* dout, float* delta,
                       int32_t row_begin, int32_t row_count, void* stream) {
    LVX_TRY(check_shape(s));
    LVX_TRY(check_tensor(o));
    LVX_TRY(check_tensor(dout));
    if (!delta) return LVX_ERR_NULL;
    LVX_TRY(check_rows(s, row_begin, row_count));
    PreParams p{};
    p.f16 = s->dtype == LVX_F16;
    p.D = s->D;
    p.o = static_cast<const uint16_t*>(o->ptr);
    p.dout = static_cast<const uint16_t*>(dout->ptr);
    p.delta = delta;
    p.os = st3(o); p.ds = st3(dout);
    p.B = s->B; p.Hq = s->Hq; p.Lq = s->Lq;
    p.row_begin = row_begin; p.row_end = row_begin + row_count;
    return static_cast<int>(launch_preprocess(p, static_cast<hipStream_t>(stream)));
}

// Work-groups of the backward are long (every step of a token block) and one
// fits a CU, so a grid that is not a multiple of the CU count wastes up to one
// whole round.  Splitting the steps of every token block over `S` work-groups evens that out.  Each leaves its fp32 sums in a slice of
// the workspace, and a launch adds a block's slices in order and rounds them; where the slices have no room, or the call accumulates,
// they are added with atomics into an fp32 scratch that is zeroed before and rounded after (or the caller's accumulator).  S minimises
//     rounds(S) * (steps / S + WG_COST) + (S > 1 ? split_cost : 0)        [in steps]
// with ranges of at least 32 steps; WG_COST is what a work-group spends outside its
// steps (operand load, ring fill, epilogue: about 8 us = 6 steps), split_cost what sharing blocks
// adds to the launch: with slices 8 and 0.3 for each of an XCD's, with atomics 55, about 70 us, measured where every block is
// shared and the whole scratch zeroed and rounded (an upper bound for a few blocks, which errs on the side of not cutting).
// lvx_bwd with atomics -> slices, us: 540 rows x 16 heads x 1346 tokens 80 -> 57.5, 3 x 500 x 12 heads of 32 x 5000 130 -> 112, 1000 x 32
// x 2000 140 -> 124, 4000 x 8 x 3000 190 -> 180, 2048 x 32 of 64 x 6404 456 -> 444, 4096 x 32 x 6404 the same.
//     rounds(S) = ceil(blocks * S / CUs)
// for equal work-groups.  With an interval mask they differ in length (a token block
// visits only the row tiles that see it; half of them is assumed); given at least two per CU the
// dispatcher fills the tail by itself and rounds(S) is the plain quotient: cutting every block then
// rarely pays (2 x 3000 rows that see the image before them: 0.98 ms in 5 ranges, added with atomics, 0.86 in none).  What fills no round is cut
// on the device there (see PlanParams).
constexpr int MAX_SLICES = 96;          // of an XCD

// How the token blocks of a launch are handed to work-groups (see bwd_kernel): per XCD, the first
// `whole` blocks get one work-group each, the next `mid` blocks `splits` work-groups each and the
// others `splits2` each.
struct BwdCut {
    int blocks_per_xcd, whole, mid, splits, splits2;
    int ranges() const { return mid * splits + (blocks_per_xcd - whole - mid) * splits2; }      // of the blocks that are cut, per XCD
    bool any_split() const { return (mid > 0 && splits > 1) || (whole + mid < blocks_per_xcd && splits2 > 1); }
};

// Every cut that is priced, the one that leaves all blocks whole first.
struct BwdCuts {
    BwdCut cut[16];
    double cost[16];
    int n;
};
static BwdCuts bwd_cuts(int blocks, int steps, bool masked, bool sliced) {
    BwdCuts all;
    all.n = 0;
    const auto add = [&](const BwdCut& cut, double cost) { all.cut[all.n] = cut; all.cost[all.n++] = cost; };
    constexpr double WG_COST = 6.0;
    const auto split_cost = [&](int ranges_per_xcd) { return sliced && ranges_per_xcd <= MAX_SLICES ? 8.0 + 0.3 * ranges_per_xcd : 55.0; };
    constexpr int XCDS = 8, MAX_SPLITS_PER_BLOCK = 16, MIN_RANGE = 32;
    const int n_cu = cu_count();
    const int per_xcd = (blocks + XCDS - 1) / XCDS;
    // unequal work-groups only even out when there are enough of them; a small masked launch
    // is priced like a dense one (which is also right when its mask hides nothing)
    const bool ragged = masked && blocks >= 2 * n_cu;
    const double work = ragged ? 0.5 * steps : (double)steps;
    for (int S = 1; S <= 8; ++S) {
        if (S > 1 && steps / S < MIN_RANGE) break;
        const double rounds = ragged ? (double)blocks * S / n_cu
                                     : (double)(((int64_t)blocks * S + n_cu - 1) / n_cu);
        const int whole = S > 1 ? 0 : per_xcd;
        add(BwdCut{per_xcd, whole, per_xcd - whole, S, 1}, rounds * (work / S + WG_COST) + (S > 1 ? split_cost(per_xcd * S) : 0.0));
    }
    // Equal blocks, more of them than CUs: whole rounds of unsplit blocks first (no partial sums,
    // one ramp per block), and only the blocks past the last whole round are cut - all alike into
    // as many ranges as fill their rounds best, or in two groups that make one round each: as
    // many blocks as give every CU one work-group when cut in S1 = ceil(CUs / blocks), and what
    // is left then in as many ranges as the CUs can take.
    const int cu_x = n_cu / XCDS;
    if (!ragged && cu_x > 0 && per_xcd > cu_x && blocks % XCDS == 0) {
        const int full = per_xcd / cu_x * cu_x, rest = per_xcd - full;
        if (rest == 0) return all;       // (whole is best then)
        const double whole_cost = (full / cu_x) * (steps + WG_COST);
        for (int S = 2; S <= 8; ++S) {
            if (steps / S < MIN_RANGE) break;
            add(BwdCut{per_xcd, full, rest, S, 1}, whole_cost + ((rest * S + cu_x - 1) / cu_x) * ((double)steps / S + WG_COST) + split_cost(rest * S));
        }
        const int S1 = (cu_x + rest - 1) / rest;
        const int n1 = std::min(rest, cu_x / S1), left = rest - n1;
        if (S1 >= 2 && steps / S1 >= MIN_RANGE && left > 0) {
            int S2 = std::min(std::min(cu_x / left, MAX_SPLITS_PER_BLOCK), steps / MIN_RANGE);
            if (S2 >= 2)
                add(BwdCut{per_xcd, full, n1, S1, S2},
                    whole_cost + ((double)steps / S1 + WG_COST) + ((double)steps / S2 + WG_COST) + split_cost(n1 * S1 + left * S2));
        }
    }
    return all;
}

static BwdCut choose_bwd_cut(int blocks, int steps, bool masked, bool sliced) {
    const BwdCuts all = bwd_cuts(blocks, steps, masked, sliced);
    int best = 0;
    for (int i = 1; i < all.n; ++i)
        if (all.cost[i] < all.cost[best]) best = i;
    return all.cut[best];
}

// The most slices an XCD can have in a window of up to so many steps: of any cut that is cheaper than none, which it is for more steps too if it
// is for these.
static int most_slices(int blocks, int steps, bool masked) {
    const BwdCuts all = bwd_cuts(blocks, steps, masked, true);
    int most = 0;
    for (int i = 1; i < all.n; ++i)
        if (all.cost[i] < all.cost[0] && all.cut[i].ranges() <= MAX_SLICES) most = std::max(most, all.cut[i].ranges());
    return most;
}

static size_t slice_bytes(const lvx_attn_shape* s) { return (size_t)2 * 128 * s->D * sizeof(float); }
static int token_blocks(const lvx_attn_shape* s) { return s->B * s->Hkv * ((s->Lkv + 127) / 128); }

// The device plans a masked launch (see PlanParams) of blocks_per_xcd token blocks that is cut nowhere.
static bool plans(const lvx_attn_shape* s, int blocks_per_xcd, int steps) {
    const int cus = cu_count() / 8;
    return s->kv_start && !s->bias && cus > 0 && cus <= 64 && blocks_per_xcd >= 2 * cus && blocks_per_xcd <= MAX_PLANNED_BLOCKS && steps >= 2 * MIN_PLANNED_RANGE;
}
static size_t plan_bytes(int slots, int shared_max) {
    return ((size_t)(8 * slots * PLAN_ENTRY + 8 * shared_max * SHARED_ENTRY) * sizeof(uint32_t) + 255) / 256 * 256;
}

// Room for fp32 sums of dK and dV: of all tokens; or, `sliced`, also of the slices that a window of up to row_count rows can have, and the plan before them.
static size_t dkv_scratch_bytes(const lvx_attn_shape* s, int32_t row_count, bool sliced) {
    const size_t all = (size_t)2 * s->B * s->Lkv * s->Hkv * s->D * sizeof(float);
    const int blocks = token_blocks(s), per_xcd = (blocks + 7) / 8, cus = cu_count() / 8;
    if (!sliced || blocks < 8 || s->Hkv <= 0 || s->Hq <= 0) return all;     // (nothing has been checked yet where only the room is asked for)
    const int steps = (int)(s->Hq / s->Hkv * (((int64_t)row_count + 31) / 32));
    size_t room = 8 * most_slices(blocks, steps, s->kv_start != nullptr) * slice_bytes(s);
    if (plans(s, per_xcd, steps)) room = std::max(room, plan_bytes(per_xcd + cus, cus) + 8 * 2 * cus * slice_bytes(s));
    return std::max(all, room);
}

static DqCut dq_cut(const lvx_attn_shape* s, int32_t row_count) {
    return dq_cut((int64_t)s->B * s->Hq, row_count, s->Lkv, s->D, cu_count());
}

// Bytes of the split contraction's partial tiles that a window of up to row_count rows can need.  Fewer rows may
// need more: a window of another 256 rows has half the splits (32 heads x 6404 tokens: 8 splits of
// 256 rows 33.6 MB, 4 of 257 18.9 MB), and a call sizes its workspace for the longest of its windows.
static size_t dq_partial_bytes(const lvx_attn_shape* s, int32_t row_count) {
    size_t most = 0;
    for (const int step : {256, 32 * DQ_FEW_TILES})
        for (int32_t r = 0; r < row_count;) {
            r = row_count - r > step ? r + step : row_count;
            const int ks = dq_splits((int64_t)s->B * s->Hq * ((r + step - 1) / step), (s->Lkv + 127) / 128, cu_count());
            if (ks <= 1) break;             // nor do longer windows split
            most = std::max(most, (size_t)ks * s->B * s->Hq * (((size_t)r + 31) / 32 * 32) * s->D * sizeof(float));
        }
    return most;
}

// Regions of the backward workspace, in order: dS^T tiles; fp32 sums of dK/dV (slices, behind the plan where there is one, or
// a scratch for atomics; with 16-bit outputs); row metadata records (2 floats per row and head); fp32 dQ partial tiles,
// one slice per split (split dQ contraction only); with an interval mask the live-tile tables (hulls of row tiles, runs
// of live tiles per token block, the groups ranked by hull length).  Every region is a multiple of 16 bytes.
struct BwdWorkspace {
    size_t ds, dkv, meta, dq32, hull, runs, order, total;
    int n_tiles, n_groups;
};

static BwdWorkspace bwd_workspace(const lvx_attn_shape* s, int32_t row_count, bool sliced) {
    BwdWorkspace w{};
    const size_t tokens = ((size_t)s->Lkv + 127) / 128 * 128;
    const size_t rows = ((size_t)row_count + 31) / 32 * 32;
    auto up16 = [](size_t n) { return (n + 15) / 16 * 16; };
    w.n_tiles = (int)(rows / 32);
    w.n_groups = (w.n_tiles + LIVE_GROUP - 1) / LIVE_GROUP;
    size_t off = 0;
    w.ds = off; off += (size_t)s->B * s->Hq * tokens * rows * sizeof(uint16_t);
    w.dkv = off; off += dkv_scratch_bytes(s, row_count, sliced);
    w.meta = off; off += (size_t)s->B * s->Hq * rows * 2 * sizeof(float);
    w.dq32 = off; off += dq_partial_bytes(s, row_count);
    if (s->kv_start) {
        const size_t nkb = tokens / 128;
        w.hull = off; off += up16((size_t)s->B * w.n_tiles * 2 * sizeof(int32_t));
        w.runs = off; off += (size_t)s->B * nkb * 8 * sizeof(int32_t);
        w.order = off; off += up16((size_t)s->B * w.n_groups * sizeof(int32_t));
    }
    w.total = off;
    return w;
}

size_t lvx_bwd_workspace_bytes(const lvx_attn_shape* s, int32_t row_count) {
    if (!s || row_count <= 0) return 0;
    return bwd_workspace(s, row_count, true).total;
}

size_t lvx_bwd_acc_workspace_bytes(const lvx_attn_shape* s, int32_t row_count) {
    if (!s || row_count <= 0) return 0;
    return bwd_workspace(s, row_count, false).total;
}

// The slices of a window's dQ that wait for the next launch to sum them.
struct WaitingDq {
    bool any;
    CastParams slices;
};

// One window, its arguments checked, in the workspace of one of ws_rows rows, at least as many, with room for slices or without.  meta: null, or the records of
// its rows.  before: null, or what the window before has left and this one may leave.
static int bwd_window(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v, const lvx_tensor* o,
                      const lvx_tensor* dout, const float* lse, const float* delta, const lvx_tensor* dq,
                      const lvx_tensor* dk, const lvx_tensor* dv, int32_t dkv_accumulate, int32_t row_begin, int32_t row_count,
                      void* workspace, int32_t ws_rows, bool sliced, hipStream_t st, const float* meta, WaitingDq* before);

// The row records' arguments.  Delta is read, or with o (and no delta) formed on the way.
static MetaParams meta_params(const lvx_attn_shape* s, const lvx_tensor* o, const lvx_tensor* dout, const float* lse, const float* delta,
                              float* out, int32_t row_begin, int32_t row_end, int n_tiles) {
    MetaParams p{lse, delta, out, s->B, s->Hq, s->Lq, row_begin, row_end, n_tiles, 1, row_end - row_begin, 0, s->scale};
    if (o) {
        p.o = static_cast<const uint16_t*>(o->ptr); p.os = st3(o);
        p.dout = static_cast<const uint16_t*>(dout->ptr); p.ds = st3(dout);
        p.D = s->D;
        p.f16 = s->dtype == LVX_F16;
    }
    return p;
}

static int bwd_impl(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v, const lvx_tensor* o,
                    const lvx_tensor* dout, const float* lse, const float* delta, const lvx_tensor* dq,
                    const lvx_tensor* dk, const lvx_tensor* dv, int32_t dkv_accumulate,
                    int32_t row_begin, int32_t row_count, void* workspace, size_t workspace_bytes, void* stream) {
    LVX_TRY(check_tensor(q));
    LVX_TRY(check_tensor(k));
    LVX_TRY(check_tensor(v));
    LVX_TRY(check_tensor(dout));
    LVX_TRY(check_tensor(dq));
    LVX_TRY(check_tensor(dk));
    LVX_TRY(check_tensor(dv));
    if (!lse) return LVX_ERR_NULL;
    const int rounds = dkv_accumulate > 0 ? dkv_accumulate >> 12 : 0;
    if (rounds > 0) dkv_accumulate &= (1 << 12) - 1;
    if (dkv_accumulate != 0 && dkv_accumulate != 1) return LVX_ERR_SHAPE;
    if (rounds > 1 && !dkv_accumulate) return LVX_ERR_SHAPE;    // 16-bit dk, dv are written by one window
    LVX_TRY(check_rows(s, row_begin, row_count));
    if (row_count == 0) return LVX_OK;
    // row offsets inside a tensor are formed in 32 bits
    if ((int64_t)s->Lq * q->stride_s >= (int64_t)1 << 31 || (int64_t)s->Lq * dout->stride_s >= (int64_t)1 << 31)
        return LVX_ERR_UNSUPPORTED;
    const int round_rows = rounds > 1 ? (row_count + rounds - 1) / rounds : row_count;
    if (!workspace || workspace_bytes < lvx_bwd_acc_workspace_bytes(s, round_rows)) return LVX_ERR_WORKSPACE;
    if (!aligned16(workspace)) return LVX_ERR_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (rounds <= 1) {
        const bool sliced = !dkv_accumulate && workspace_bytes >= lvx_bwd_workspace_bytes(s, row_count);
        return bwd_window(s, q, k, v, o, dout, lse, delta, dq, dk, dv, dkv_accumulate, row_begin, row_count, workspace, row_count, sliced, st, nullptr, nullptr);
    }

    // Several windows: the records of all their rows by one launch instead of one of 3 - 5 us each (32 heads x 16 rounds of 256 rows,
    // forward and backward 2775 -> 2741 us), where the scratch that only sums of 16-bit dk, dv use holds them.
    const int n = (row_count + round_rows - 1) / round_rows;
    const BwdWorkspace w = bwd_workspace(s, round_rows, false);
    const int64_t each = (int64_t)s->B * s->Hq * w.n_tiles * 64;
    float* meta = nullptr;
    if (n <= 65535 && (size_t)each * n * sizeof(float) <= w.meta - w.dkv) {
        meta = reinterpret_cast<float*>(static_cast<char*>(workspace) + w.dkv);
        MetaParams mp = meta_params(s, o, dout, lse, delta, meta, row_begin, row_begin + row_count, w.n_tiles);
        mp.rounds = n; mp.round_rows = round_rows; mp.round_out = each;
        const hipError_t e = launch_bwd_meta(mp, st);
        if (e != hipSuccess) return static_cast<int>(e);
    }
    WaitingDq waiting{};
    for (int r = 0; r < n; ++r)
        LVX_TRY(bwd_window(s, q, k, v, o, dout, lse, delta, dq, dk, dv, 1, row_begin + r * round_rows, std::min(round_rows, row_count - r * round_rows),
                           workspace, round_rows, false, st, meta ? meta + r * each : nullptr, &waiting));
    return waiting.any ? static_cast<int>(launch_cast(waiting.slices, st)) : LVX_OK;
}

int lvx_bwd(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v,
            const lvx_tensor* dout, const float* lse, const float* delta, const lvx_tensor* dq,
            const lvx_tensor* dk, const lvx_tensor* dv, int32_t dkv_accumulate,
            int32_t row_begin, int32_t row_count, void* workspace, size_t workspace_bytes, void* stream) {
    LVX_TRY(check_shape(s));
    if (!delta) return LVX_ERR_NULL;
    return bwd_impl(s, q, k, v, nullptr, dout, lse, delta, dq, dk, dv, dkv_accumulate, row_begin, row_count, workspace, workspace_bytes, stream);
}

int lvx_bwd_from_o(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v, const lvx_tensor* o,
                   const lvx_tensor* dout, const float* lse, const lvx_tensor* dq, const lvx_tensor* dk, const lvx_tensor* dv,
                   int32_t dkv_accumulate, int32_t row_begin, int32_t row_count, void* workspace, size_t workspace_bytes, void* stream) {
    LVX_TRY(check_shape(s));
    LVX_TRY(check_tensor(o));
    return bwd_impl(s, q, k, v, o, dout, lse, nullptr, dq, dk, dv, dkv_accumulate, row_begin, row_count, workspace, workspace_bytes, stream);
}

static int bwd_window(const lvx_attn_shape* s, const lvx_tensor* q, const lvx_tensor* k, const lvx_tensor* v, const lvx_tensor* o,
                      const lvx_tensor* dout, const float* lse, const float* delta, const lvx_tensor* dq,
                      const lvx_tensor* dk, const lvx_tensor* dv, int32_t dkv_accumulate, int32_t row_begin, int32_t row_count,
                      void* workspace, int32_t ws_rows, bool sliced, hipStream_t st, const float* meta, WaitingDq* before) {
    BwdParams p{};
    p.f16 = s->dtype == LVX_F16;
    p.D = s->D;
    p.q = static_cast<const uint16_t*>(q->ptr);
    p.k = static_cast<const uint16_t*>(k->ptr);
    p.v = static_cast<const uint16_t*>(v->ptr);
    p.dout = static_cast<const uint16_t*>(dout->ptr);
    p.dk = dk->ptr; p.dv = dv->ptr;
    p.qs = st3(q); p.ks = st3(k); p.vs = st3(v); p.dos = st3(dout); p.dks = st3(dk); p.dvs = st3(dv);
    p.kv_len = s->kv_len; p.kv_start = s->kv_start; p.kv_end = s->kv_end;
    p.bias = s->bias; p.bias_b = s->bias_stride_b; p.bias_h = s->bias_stride_h; p.bias_r = s->bias_stride_r;
    p.B = s->B; p.Hq = s->Hq; p.Hkv = s->Hkv; p.Lq = s->Lq; p.Lkv = s->Lkv; p.G = s->Hq / s->Hkv;
    p.row_begin = row_begin; p.row_end = row_begin + row_count;
    p.n_kv_blocks = (s->Lkv + 127) / 128;
    p.scale = s->scale; p.scale_log2e = s->scale * LOG2E;
    const int64_t tokens = (int64_t)p.n_kv_blocks * 128;
    const int64_t rows = ((int64_t)row_count + 31) / 32 * 32;
    p.ds_ws = static_cast<uint16_t*>(workspace);
    p.ws_ld = rows * 128;          // one token block: (rows / 32) tiles of 128 x 32
    p.ws_bh = tokens * rows;
    // dS^T is written once and read once.  Where it does not fit the memory-side cache (256 MB) it should not
    // push out of the caches what is read again (Q and dO tiles by the token blocks of a head, K by the dQ
    // kernel): streaming stores, streaming loads.  us, forward + backward, without and with: 6404 tokens x 4096 rows x
    // 32 heads (1.7 GB) 1879 -> 1821, x 1024 rows (0.4 GB) 794 -> 774, heads of 64 x 2048 rows (0.8 GB) 676 ->
    // 595, 2 x 3000 rows with image intervals 1205 -> 1152.  Where it fits, the hint costs a little: x 512 rows of
    // heads of 64 (0.2 GB) 208 -> 213, rounds of 256 rows (0.1 GB) 2940 -> 2966 for sixteen.
    p.ds_stream = (int64_t)s->B * s->Hq * p.ws_bh * 2 > ((int64_t)240 << 20);

    const BwdWorkspace wsl = bwd_workspace(s, ws_rows, sliced);
    const int n_tiles = (int)(rows / 32), n_groups = (n_tiles + LIVE_GROUP - 1) / LIVE_GROUP;
    char* const wsb = static_cast<char*>(workspace);
    // how the launch is shaped decides which fp32 scratches it accumulates into; the
    // metadata kernel zeroes them on its way
    const int blocks = s->B * s->Hkv * p.n_kv_blocks;
    const int steps = p.G * (int)(rows / 32);
    const BwdCut cut = choose_bwd_cut(blocks, steps, s->kv_start != nullptr, blocks >= 8 && sliced);
    if (cut.any_split() && sliced && (size_t)8 * cut.ranges() * slice_bytes(s) <= wsl.meta - wsl.dkv) {
        p.slices = reinterpret_cast<float*>(wsb + wsl.dkv);
        p.per_xcd = cut.ranges();
    }
    // With intervals per row how long a block is shows on the device, which then plans the launch, in the fp32 scratch.  (A bias
    // seldom hides anything, and the plan would be 3 us for nothing.)
    PlanParams plan{};
    const int cus = cu_count() / 8;
    if (plans(s, cut.blocks_per_xcd, steps) && !meta && !dkv_accumulate && !cut.any_split() && (int64_t)s->B * n_groups * LIVE_GROUP <= MAX_LIVE_TILES) {
        plan.cus = plan.shared_max = cus;
        plan.slots = cut.blocks_per_xcd + cus;
        plan.n_blocks = blocks; plan.blocks_per_xcd = cut.blocks_per_xcd; plan.G = p.G;
        plan.entries = reinterpret_cast<uint32_t*>(wsb + wsl.dkv);
        plan.shared = plan.entries + 8 * plan.slots * PLAN_ENTRY;
        const size_t tables = plan_bytes(plan.slots, plan.shared_max);
        const size_t room = wsl.meta - wsl.dkv;
        plan.slices = room > tables ? (int)std::min<size_t>((room - tables) / slice_bytes(s) / 8, 2 * cus) : 0;
        if (plan.slices < 2) plan.entries = nullptr;
        else p.slices = reinterpret_cast<float*>(wsb + wsl.dkv + tables);
        p.plan = plan.entries;
        if (plan.entries) p.per_xcd = plan.slots;
    }
    p.n_blocks = blocks;
    p.blocks_per_xcd = cut.blocks_per_xcd;
    p.whole_blocks = cut.whole;
    p.mid_blocks = cut.mid;
    p.q_splits = cut.splits;
    p.q_splits2 = cut.splits2;
    p.dkv_mode = cut.any_split() && !p.slices ? 2 : (dkv_accumulate ? 1 : 0);
    float* const scratch = p.dkv_mode == 2 && !dkv_accumulate ? reinterpret_cast<float*>(wsb + wsl.dkv) : nullptr;
    const DqCut dq_by = dq_cut(s, row_count);
    float* const dq32 = dq_by.splits > 1 ? reinterpret_cast<float*>(wsb + wsl.dq32) : nullptr;
    // the token blocks several work-groups share, and the fp32 scratch of the call that sums them
    SharedBlocks sb{s->B, s->Hkv, s->Lkv, s->D, p.n_kv_blocks, p.n_blocks, p.blocks_per_xcd, p.whole_blocks};
    int32_t* hull = nullptr;
    int32_t* order = nullptr;
    LiveParams lp{};
    if (s->kv_start) {
        // interval mask: token blocks skip the row tiles that see none of their tokens
        hull = reinterpret_cast<int32_t*>(wsb + wsl.hull);
        // the ranking is quadratic in the number of groups; where there are that many, the dQ
        // kernel's work-groups even out in index order
        if (!dq_by.few && dq_by.splits <= 1 && s->B * n_groups <= MAX_RANKED_GROUPS) order = reinterpret_cast<int32_t*>(wsb + wsl.order);
        lp = LiveParams{s->kv_len, s->kv_start, s->kv_end, hull, reinterpret_cast<int32_t*>(wsb + wsl.runs), order,
                        s->B, s->Lq, s->Lkv, row_begin,
                        row_begin + row_count, n_tiles, n_groups, p.n_kv_blocks, plan};
        p.live_runs = lp.live_runs;
    }
    const bool has_hulls = !meta;       // its records come by a launch of its own, which writes the tables as well, or their hulls
    if (!meta) {
        float* const out = reinterpret_cast<float*>(wsb + wsl.meta);
        MetaParams mp = meta_params(s, o, dout, lse, delta, out, row_begin, row_begin + row_count, n_tiles);
        mp.scratch = scratch;
        mp.sb = sb;
        hipError_t em = launch_bwd_meta(mp, st, hull ? &lp : nullptr);
        if (em != hipSuccess) return static_cast<int>(em);
        meta = out;
    }
    p.meta = meta;
    if (hull) {
        hipError_t el = launch_bwd_live(lp, st, has_hulls);
        if (el != hipSuccess) return static_cast<int>(el);
    }

    const int64_t dkv_elems = (int64_t)s->B * s->Lkv * s->Hkv * s->D;
    // blocks with one work-group are written by it as the caller asked
    p.dk_whole = p.dk; p.dv_whole = p.dv;
    p.dks_whole = p.dks; p.dvs_whole = p.dvs;
    p.whole_mode = dkv_accumulate ? 1 : 0;
    if (scratch) {
        // bf16 outputs, several work-groups per token block: those blocks are summed in the fp32
        // scratch [2][B, Lkv, Hkv, D] and rounded once afterwards
        p.dk = scratch;
        p.dv = scratch + dkv_elems;
        p.dks = p.dvs = Strides3{(int64_t)s->Lkv * s->Hkv * s->D, (int64_t)s->D, (int64_t)s->Hkv * s->D};
    }
    // (the slices lie where this window's own come, which only the launch after this one writes)
    hipError_t e = launch_bwd(p, s->kv_start != nullptr, st, before && before->any ? &before->slices : nullptr);
    if (e != hipSuccess) return static_cast<int>(e);
    if (before) before->any = false;
    if (scratch) {
        CastSharedParams cp{sb, scratch, static_cast<uint16_t*>(dk->ptr), static_cast<uint16_t*>(dv->ptr), st3(dk), st3(dv), p.f16};
        e = launch_cast_shared(cp, st);
        if (e != hipSuccess) return static_cast<int>(e);
    }

    CastSlicesParams cp{};
    bool rides = false;
    if (p.slices) {
        cp = CastSlicesParams{plan.entries ? plan.shared : nullptr, plan.entries ? plan.shared_max : cut.blocks_per_xcd - cut.whole,
                              cut.whole, cut.mid, cut.splits, cut.splits2, p.per_xcd, blocks, cut.blocks_per_xcd,
                              p.slices, s->B, s->Lkv, s->D, p.n_kv_blocks, p.f16, static_cast<uint16_t*>(dk->ptr),
                              static_cast<uint16_t*>(dv->ptr), st3(dk), st3(dv)};
        // In the launch of dQ where there are few of them: its work-groups have a CU's registers to themselves or share them with one
        // other, and more than a round of the slices' would keep it waiting.  lvx_bwd, a launch of its own -> in dQ's, us: 540 rows x 16
        // heads x 1346 tokens (192 work-groups) 58.7 -> 54.0, 2378 x 64 of 64 x 700 159.8 -> 154.3; 3 x 500 x 12 of 32 x 5000 (416) would go
        // 112 -> 120, 2048 x 32 of 64 x 6404 (608) 439 -> 469.
        rides = cast_slices_blocks(cp) <= cu_count();
        if (!rides) {
            e = launch_cast_slices(cp, st);
            if (e != hipSuccess) return static_cast<int>(e);
        }
    }

    // dQ[b, h, rows, :] = dS^T[b, h]^T (rows x tokens) * K[b, h / G] (tokens x D), scale already in dS
    DqParams g{};
    g.ds = p.ds_ws; g.ds_bh = p.ws_bh;
    g.k = p.k; g.ks = p.ks;
    g.dq = static_cast<uint16_t*>(dq->ptr) + (int64_t)row_begin * dq->stride_s;
    g.dqs = st3(dq);
    g.B = s->B; g.Hq = s->Hq; g.G = p.G; g.D = s->D; g.f16 = p.f16;
    g.rows = row_count; g.row_tiles = (int)(rows / 32); g.Lkv = s->Lkv;
    g.stream = p.ds_stream;
    g.kv_len = s->kv_len;
    g.tile_range = hull;         // [B][row tiles][2]
    g.order = order;
    g.few = dq_by.few;
    // split contraction: every split stores its partial tiles in its own fp32 slice; the
    // cast sums the slices and rounds into dq
    g.k_splits = dq_by.splits; g.split_len = dq_by.split_len;
    g.part = dq32; g.part_split = (int64_t)s->B * s->Hq * row_count * s->D;      // [split][B * Hq][D][row_count]
    e = launch_dq(g, st, rides ? &cp : nullptr);
    if (e != hipSuccess || dq_by.splits <= 1) return static_cast<int>(e);
    CastParams cq{};
    cq.f16 = p.f16;
    cq.D = s->D;
    cq.src = dq32;
    cq.dst = static_cast<uint16_t*>(dq->ptr) + (int64_t)row_begin * dq->stride_s;
    cq.ds = st3(dq);
    cq.B = s->B; cq.H = s->Hq; cq.L = row_count;
    cq.transposed = 1;
    cq.nsum = dq_by.splits; cq.sum_stride = g.part_split;
    if (before) {
        *before = WaitingDq{true, cq};
        return LVX_OK;
    }
    return static_cast<int>(launch_cast(cq, st));
}

static int check_dtype(int32_t dtype) { return (dtype == LVX_BF16 || dtype == LVX_F16) ? LVX_OK : LVX_ERR_DTYPE; }

int lvx_cast_f32(const float* src, const lvx_tensor* dst, int32_t B, int32_t H, int32_t L, int32_t D,
                 int32_t dtype, void* stream) {
    LVX_TRY(check_dtype(dtype));
    if (!src) return LVX_ERR_NULL;
    LVX_TRY(check_tensor(dst));
    if (!aligned16(src)) return LVX_ERR_ALIGN;
    if (D != 128 && D != 64 && D != 32 && D != 16) return LVX_ERR_HEAD_DIM;
    if (B <= 0 || H <= 0 || L <= 0) return LVX_ERR_SHAPE;
    CastParams p{};
    p.f16 = dtype == LVX_F16;
    p.D = D;
    p.src = src;
    p.dst = static_cast<uint16_t*>(dst->ptr);
    p.ds = st3(dst);
    p.B = B; p.H = H; p.L = L;
    return static_cast<int>(launch_cast(p, static_cast<hipStream_t>(stream)));
}

static int check_gemm_ptr(const void* p, int64_t ld) {
    if (!p) return LVX_ERR_NULL;
    if (!aligned16(p) || (ld % 8) != 0) return LVX_ERR_ALIGN;
    if (ld <= 0 || ld >= (1 << 21)) return LVX_ERR_SHAPE;   // 32-bit byte offsets inside a tile
    return LVX_OK;
}

}  // extern "C"

static void fill_grid(GemmParams& g, int M, int N, int nprob) { g.M = M; g.N = N; g.nprob = nprob; }

extern "C" {

static int kv_proj_impl(const void* x, int64_t ldx, const void* w_k, const void* w_v, int64_t ldw, int32_t w_in_major,
                        void* k_out, void* v_out, int64_t ldkv, int32_t M, int32_t Dm, int32_t N,
                        const void* k_norm_w, float eps, void* k_raw, float* k_rstd, int32_t dtype, void* stream) {
    LVX_TRY(check_dtype(dtype));
    LVX_TRY(check_gemm_ptr(x, ldx));
    LVX_TRY(check_gemm_ptr(w_k, ldw));
    LVX_TRY(check_gemm_ptr(k_out, ldkv));
    if (!w_v != !v_out) return LVX_ERR_NULL;       // both or neither
    const int np = w_v ? 2 : 1;                    // one projection only: the Q side
    if (np == 2) {
        LVX_TRY(check_gemm_ptr(w_v, ldw));
        LVX_TRY(check_gemm_ptr(v_out, ldkv));
    }
    if (M <= 0 || Dm <= 0 || N <= 0 || (Dm % 8) || (N % 8)) return LVX_ERR_SHAPE;
    if (ldx < Dm || ldkv < N || ldw < (w_in_major ? N : Dm)) return LVX_ERR_SHAPE;
    GemmParams g{};
    g.f16 = dtype == LVX_F16;
    const void* w[2] = {w_k, w_v};
    void* c[2] = {k_out, v_out};
    for (int i = 0; i < np; ++i) {
        GemmProblem& pr = g.prob[i];
        pr.A[0] = static_cast<const uint16_t*>(x); pr.lda[0] = ldx;
        pr.Bm[0] = static_cast<const uint16_t*>(w[i]); pr.ldb[0] = ldw;
        pr.K[0] = Dm; pr.nseg = 1;
        pr.C = static_cast<uint16_t*>(c[i]); pr.ldc = ldkv;
    }
    if (k_norm_w) {
        if (N % 128) return LVX_ERR_HEAD_DIM;      // the norm runs over heads of 128 columns
        if (!aligned16(k_norm_w)) return LVX_ERR_ALIGN;
        if (!(eps >= 0.f)) return LVX_ERR_SHAPE;
        if (k_raw) LVX_TRY(check_gemm_ptr(k_raw, ldkv));
        if (k_rstd && (reinterpret_cast<uintptr_t>(k_rstd) & 3)) return LVX_ERR_ALIGN;
        g.norm_w = static_cast<const uint16_t*>(k_norm_w);
        g.norm_eps = eps;
        g.c_raw = static_cast<uint16_t*>(k_raw);
        g.rstd = k_rstd;
    }
    fill_grid(g, M, N, np);
    return static_cast<int>(launch_gemm(g, false, w_in_major != 0, static_cast<hipStream_t>(stream)));
}

int lvx_kv_proj(const void* x, int64_t ldx, const void* w_k, const void* w_v, int64_t ldw, int32_t w_in_major,
                void* k_out, void* v_out, int64_t ldkv, int32_t M, int32_t Dm, int32_t N, int32_t dtype, void* stream) {
    return kv_proj_impl(x, ldx, w_k, w_v, ldw, w_in_major, k_out, v_out, ldkv, M, Dm, N, nullptr, 0.f, nullptr,
                        nullptr, dtype, stream);
}

int lvx_kv_proj_norm(const void* x, int64_t ldx, const void* w_k, const void* w_v, int64_t ldw, int32_t w_in_major,
                     void* k_out, void* v_out, int64_t ldkv, int32_t M, int32_t Dm, int32_t N,
                     const void* k_norm_w, float eps, void* k_raw, float* k_rstd, int32_t dtype, void* stream) {
    if (!k_norm_w) return LVX_ERR_NULL;
    return kv_proj_impl(x, ldx, w_k, w_v, ldw, w_in_major, k_out, v_out, ldkv, M, Dm, N, k_norm_w, eps, k_raw,
                        k_rstd, dtype, stream);
}

int lvx_k_norm_bwd(const void* dk, int64_t lddk, const void* k_raw, int64_t ldk, const float* k_rstd,
                   const void* k_norm_w, void* dk_raw, int64_t lddk_raw, float* dw, int32_t M, int32_t N,
                   int32_t dtype, void* stream) {
    LVX_TRY(check_dtype(dtype));
    LVX_TRY(check_gemm_ptr(dk, lddk));
    LVX_TRY(check_gemm_ptr(k_raw, ldk));
    LVX_TRY(check_gemm_ptr(dk_raw, lddk_raw));
    if (!k_rstd || !k_norm_w) return LVX_ERR_NULL;
    if (!aligned16(k_norm_w) || (reinterpret_cast<uintptr_t>(k_rstd) & 3) || (reinterpret_cast<uintptr_t>(dw) & 3))
        return LVX_ERR_ALIGN;
    if (M <= 0 || N <= 0) return LVX_ERR_SHAPE;
    if (N % 128) return LVX_ERR_HEAD_DIM;
    if (lddk < N || ldk < N || lddk_raw < N) return LVX_ERR_SHAPE;
    NormBwdParams p{};
    p.f16 = dtype == LVX_F16;
    p.dy = static_cast<const uint16_t*>(dk);
    p.x = static_cast<const uint16_t*>(k_raw);
    p.rstd = k_rstd;
    p.w = static_cast<const uint16_t*>(k_norm_w);
    p.dx = static_cast<uint16_t*>(dk_raw);
    p.dw = dw;
    p.ldy = lddk; p.ldx = ldk; p.lddx = lddk_raw;
    p.M = M; p.heads = N / 128;
    return static_cast<int>(launch_norm_bwd(p, static_cast<hipStream_t>(stream)));
}

int lvx_dx_vis(const void* dk, const void* dv, int64_t lddkv, const void* w_k, const void* w_v, int64_t ldw,
               int32_t w_in_major, void* dx, int64_t lddx, int32_t M, int32_t Dm, int32_t N, int32_t dtype,
               void* stream) {
    LVX_TRY(check_dtype(dtype));
    LVX_TRY(check_gemm_ptr(dk, lddkv));
    LVX_TRY(check_gemm_ptr(w_k, ldw));
    LVX_TRY(check_gemm_ptr(dx, lddx));
    if (!dv != !w_v) return LVX_ERR_NULL;          // both or neither
    if (dv) {
        LVX_TRY(check_gemm_ptr(dv, lddkv));
        LVX_TRY(check_gemm_ptr(w_v, ldw));
    }
    if (M <= 0 || Dm <= 0 || N <= 0 || (Dm % 8) || (N % 8)) return LVX_ERR_SHAPE;
    if (lddkv < N || lddx < Dm || ldw < (w_in_major ? N : Dm)) return LVX_ERR_SHAPE;
    GemmParams g{};
    g.f16 = dtype == LVX_F16;
    GemmProblem& pr = g.prob[0];
    pr.A[0] = static_cast<const uint16_t*>(dk); pr.A[1] = static_cast<const uint16_t*>(dv);
    pr.lda[0] = pr.lda[1] = lddkv;
    pr.Bm[0] = static_cast<const uint16_t*>(w_k); pr.Bm[1] = static_cast<const uint16_t*>(w_v);
    pr.ldb[0] = pr.ldb[1] = ldw;
    pr.K[0] = N; pr.K[1] = dv ? N : 0; pr.nseg = dv ? 2 : 1;
    pr.C = static_cast<uint16_t*>(dx); pr.ldc = lddx;
    fill_grid(g, M, Dm, 1);
    // B[k = n][col = dm]: W [Dm][N] has k contiguous, W [N][Dm] has the column contiguous
    return static_cast<int>(launch_gemm(g, false, w_in_major == 0, static_cast<hipStream_t>(stream)));
}

int lvx_dw_kv(const void* x, int64_t ldx, const void* dk, const void* dv, int64_t lddkv, void* dw_k, void* dw_v,
              int64_t ldw, int32_t w_in_major, int32_t M, int32_t Dm, int32_t N, int32_t dtype, void* stream) {
    LVX_TRY(check_dtype(dtype));
    LVX_TRY(check_gemm_ptr(x, ldx));
    LVX_TRY(check_gemm_ptr(dk, lddkv));
    LVX_TRY(check_gemm_ptr(dw_k, ldw));
    if (!dv != !dw_v) return LVX_ERR_NULL;         // both or neither
    const int np = dv ? 2 : 1;
    if (np == 2) {
        LVX_TRY(check_gemm_ptr(dv, lddkv));
        LVX_TRY(check_gemm_ptr(dw_v, ldw));
    }
    if (M <= 0 || Dm <= 0 || N <= 0 || (Dm % 8) || (N % 8)) return LVX_ERR_SHAPE;
    if (ldx < Dm || lddkv < N || ldw < (w_in_major ? N : Dm)) return LVX_ERR_SHAPE;
    GemmParams g{};
    g.f16 = dtype == LVX_F16;
    const void* d[2] = {dk, dv};
    void* c[2] = {dw_k, dw_v};
    for (int i = 0; i < np; ++i) {
        GemmProblem& pr = g.prob[i];
        if (w_in_major) {   // dW [Dm][N] = X^T dK
            pr.A[0] = static_cast<const uint16_t*>(x); pr.lda[0] = ldx;
            pr.Bm[0] = static_cast<const uint16_t*>(d[i]); pr.ldb[0] = lddkv;
        } else {            // dW [N][Dm] = dK^T X
            pr.A[0] = static_cast<const uint16_t*>(d[i]); pr.lda[0] = lddkv;
            pr.Bm[0] = static_cast<const uint16_t*>(x); pr.ldb[0] = ldx;
        }
        pr.K[0] = M; pr.nseg = 1;
        pr.C = static_cast<uint16_t*>(c[i]); pr.ldc = ldw;
    }
    if (w_in_major) fill_grid(g, Dm, N, np);
    else fill_grid(g, N, Dm, np);
    return static_cast<int>(launch_gemm(g, true, true, static_cast<hipStream_t>(stream)));
}

}  // extern "C"

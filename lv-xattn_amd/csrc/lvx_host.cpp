// The per-call host work of the attention operators in native code: what ops.py and attn.py would
// otherwise do with some forty Python and ctypes operations a call (argument checks, tensor descriptions,
// the current stream, output and workspace tensors).  A decoded token's two launches take 12 us on the
// GPU; issuing them through ctypes took 32 us of host time.
//
// The library's functions are those of the liblvx.so that the package has loaded, handed over by address
// (bind): this module is linked to none.
//
// An operator answers False, and queues nothing, when a call is not one it can pass on as it is (a wrong
// type, shape or device among the arguments); the caller then goes through its own checks, which word
// the error.
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <map>
#include <optional>
#include <string>

#include "../../include/lvx.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

struct Library {
    decltype(&lvx_fwd_workspace_bytes) fwd_workspace_bytes;
    decltype(&lvx_fwd) fwd;
    decltype(&lvx_fwd_acc) fwd_acc;
    decltype(&lvx_bwd_preprocess) bwd_preprocess;
    decltype(&lvx_bwd) bwd;
    decltype(&lvx_bwd_from_o) bwd_from_o;
    decltype(&lvx_bwd_workspace_bytes) bwd_workspace_bytes, bwd_acc_workspace_bytes;
    decltype(&lvx_bias_hull) bias_hull;
} lib;

void bind(const std::map<std::string, uintptr_t>& addresses) {
    auto set = [&](auto& f, const char* name) { f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(addresses.at(name)); };
    set(lib.fwd_workspace_bytes, "lvx_fwd_workspace_bytes");
    set(lib.fwd, "lvx_fwd");
    set(lib.fwd_acc, "lvx_fwd_acc");
    set(lib.bwd_preprocess, "lvx_bwd_preprocess");
    set(lib.bwd, "lvx_bwd");
    set(lib.bwd_from_o, "lvx_bwd_from_o");
    set(lib.bwd_workspace_bytes, "lvx_bwd_workspace_bytes");
    set(lib.bwd_acc_workspace_bytes, "lvx_bwd_acc_workspace_bytes");
    set(lib.bias_hull, "lvx_bias_hull");
}

int dtype_code(const Tensor& t) {
    return t.scalar_type() == at::kBFloat16 ? LVX_BF16 : t.scalar_type() == at::kHalf ? LVX_F16 : 0;
}

lvx_tensor t4(const Tensor& t) { return lvx_tensor{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

// a 4-d tensor on q's device with unit last stride
bool plain4(const Tensor& t, const Tensor& q, at::ScalarType type) {
    return t.dim() == 4 && t.stride(3) == 1 && t.scalar_type() == type && t.device() == q.device();
}

bool rows_ok(const Tensor& l, const Tensor& q) {        // LSE, delta: contiguous fp32 [B * Hq, Lq]
    return l.scalar_type() == at::kFloat && l.is_contiguous() && l.numel() == q.size(0) * q.size(1) * q.size(2) && l.device() == q.device();
}

bool mask_ok(const OptTensor& m, const Tensor& q, bool per_row) {
    if (!m) return true;
    return m->scalar_type() == at::kInt && m->device() == q.device() && m->is_contiguous() && m->dim() == (per_row ? 2 : 1) &&
           m->size(0) == q.size(0) && (!per_row || m->size(1) == q.size(2));
}

// Fills the shape from tensors of one type and device; false when something does not fit.
bool fill_shape(lvx_attn_shape& s, const Tensor& q, const Tensor& k, const Tensor& v, double scale, const OptTensor& kv_len,
                const OptTensor& kv_start, const OptTensor& kv_end) {
    const int dt = dtype_code(q);
    if (!q.is_cuda() || !dt || !plain4(q, q, q.scalar_type()) || !plain4(k, q, q.scalar_type()) || !plain4(v, q, q.scalar_type()))
        return false;
    if (k.size(0) != q.size(0) || k.size(3) != q.size(3) || v.sizes() != k.sizes()) return false;
    if (!mask_ok(kv_len, q, false) || !mask_ok(kv_start, q, true) || !mask_ok(kv_end, q, true) || !kv_start != !kv_end) return false;
    if (c10::hip::current_device() != q.device().index()) return false;       // launches go to the current device
    s = lvx_attn_shape{};
    s.B = (int32_t)q.size(0); s.Hq = (int32_t)q.size(1); s.Hkv = (int32_t)k.size(1); s.D = (int32_t)q.size(3);
    s.Lq = (int32_t)q.size(2); s.Lkv = (int32_t)k.size(2); s.dtype = dt; s.scale = (float)scale;
    if (kv_len) s.kv_len = kv_len->data_ptr<int32_t>();
    if (kv_start) { s.kv_start = kv_start->data_ptr<int32_t>(); s.kv_end = kv_end->data_ptr<int32_t>(); }
    return true;
}

// The dense bias of a call, fp32 [B|1, Hq|1, Lq, Lkv]; false when the library would refuse it.  A dimension of extent
// 1 is never stepped over: the library is told the stride its own checks accept, whatever the tensor says.
bool fill_bias(lvx_attn_shape& s, const OptTensor& bias, const Tensor& q) {
    if (!bias) return true;
    const Tensor& t = *bias;
    if (!plain4(t, q, at::kFloat) || (t.size(0) != 1 && t.size(0) != s.B) || (t.size(1) != 1 && t.size(1) != s.Hq) || t.size(2) != s.Lq ||
        t.size(3) != s.Lkv)
        return false;
    const int64_t row = ((int64_t)s.Lkv + 3) / 4 * 4;
    s.bias = t.data_ptr<float>();
    s.bias_stride_b = t.size(0) > 1 ? t.stride(0) : 0;
    s.bias_stride_h = t.size(1) > 1 ? t.stride(1) : 0;
    s.bias_stride_r = s.Lq > 1 ? t.stride(2) : row;
    return s.bias_stride_r >= row && !((s.bias_stride_b | s.bias_stride_h | s.bias_stride_r) & 3) &&
           !(reinterpret_cast<uintptr_t>(s.bias) & 15);
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// Calls the library without the interpreter's lock - a launch may block on a full queue, and other Python threads go
// on meanwhile, as they do through ctypes - and gives its code as the package's own exception.
template <typename F>
void call(const char* what, F f) {
    int rc;
    {
        py::gil_scoped_release unlocked;
        rc = f();
    }
    if (rc) py::module_::import("lv_xattn._lib").attr("check")(rc, what);
}

// Whether the kernels can read every one of these where it lies: unit last stride, the others multiples
// of 8 elements, 16-byte aligned.
bool usable(const Tensor& a, const Tensor& b, const Tensor& c) {
    for (const Tensor* t : {&a, &b, &c})
        if (t->dim() != 4 || t->stride(3) != 1 || ((t->stride(0) | t->stride(1) | t->stride(2)) & 7) ||
            (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15))
            return false;
    return true;
}

// (o, lse, workspace or None) of a forward: o like q and contiguous, or the view of [B, Lq, Hq, D] memory with
// `token_major`; lse fp32 [B * Hq, Lq]; room for the parts of kv_splits key splits over `rows` rows, of rounds in one call where
// k says how many keys there are and `biased` whether with a dense bias.
py::tuple round_buffers(const Tensor& q, int64_t rows, int64_t kv_splits, bool token_major, const OptTensor& k, bool biased) {
    const int64_t B = q.size(0), H = q.size(1), L = q.size(2), D = q.size(3);
    Tensor o = token_major ? at::empty({B, L, H, D}, q.options()).transpose(1, 2) : at::empty({B, H, L, D}, q.options());
    Tensor lse = at::empty({B * H, L}, q.options().dtype(at::kFloat));
    if (kv_splits <= 1) return py::make_tuple(std::move(o), std::move(lse), py::none());
    lvx_attn_shape s{};
    s.B = (int32_t)B; s.Hq = (int32_t)H; s.D = (int32_t)D;
    if (k) { s.Hkv = (int32_t)k->size(1); s.Lkv = (int32_t)k->size(2); }
    if (biased) s.bias = lse.data_ptr<float>();         // only whether there is one matters
    Tensor ws = at::empty({(int64_t)lib.fwd_workspace_bytes(&s, (int32_t)rows, (int32_t)kv_splits)}, q.options().dtype(at::kByte));
    return py::make_tuple(std::move(o), std::move(lse), std::move(ws));
}

// The same of a single launch, whose caller (a decoded token waits for the host) does not ask for more than it needs.
py::tuple forward_buffers(const Tensor& q, int64_t rows, int64_t kv_splits, bool token_major) {
    return round_buffers(q, rows, kv_splits, token_major, {}, false);
}

bool fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, double scale, int64_t row_begin,
         int64_t row_count, const OptTensor& kv_len, const OptTensor& kv_start, const OptTensor& kv_end, int64_t kv_splits,
         const OptTensor& ws, const OptTensor& acc_o, const OptTensor& acc_l, const OptTensor& bias) {
    lvx_attn_shape s;
    if (!fill_shape(s, q, k, v, scale, kv_len, kv_start, kv_end) || !fill_bias(s, bias, q) || !plain4(o, q, q.scalar_type()) || o.sizes() != q.sizes() || !rows_ok(lse, q))
        return false;
    const lvx_tensor tq = t4(q), tk = t4(k), tv = t4(v), to = t4(o);
    void* const wp = ws ? ws->data_ptr() : nullptr;
    const size_t wb = ws ? ws->nbytes() : 0;
    float* const lp = lse.data_ptr<float>();
    void* const st = current_stream();
    if (!acc_o) {
        call("lvx_fwd", [&] {
            return lib.fwd(&s, &tq, &tk, &tv, &to, lp, (int32_t)row_begin, (int32_t)row_count, (int32_t)kv_splits, wp, wb, st);
        });
        return true;
    }
    if (!plain4(*acc_o, q, q.scalar_type()) || acc_o->sizes() != q.sizes() || !acc_l || !rows_ok(*acc_l, q)) return false;
    const lvx_tensor ta = t4(*acc_o);
    const float* const la = acc_l->data_ptr<float>();
    call("lvx_fwd_acc", [&] {
        return lib.fwd_acc(&s, &tq, &tk, &tv, &ta, la, &to, lp, (int32_t)row_begin, (int32_t)row_count, (int32_t)kv_splits, wp, wb, st);
    });
    return true;
}

bool bwd_preprocess(const Tensor& o, const Tensor& dout, const Tensor& delta, int64_t row_begin, int64_t row_count) {
    lvx_attn_shape s;
    if (!fill_shape(s, o, dout, dout, 1.0, {}, {}, {}) || o.sizes() != dout.sizes() || !rows_ok(delta, o)) return false;
    const lvx_tensor to = t4(o), td = t4(dout);
    float* const dp = delta.data_ptr<float>();
    void* const st = current_stream();
    call("lvx_bwd_preprocess", [&] { return lib.bwd_preprocess(&s, &to, &td, dp, (int32_t)row_begin, (int32_t)row_count, st); });
    return true;
}

// delta, or the o to form it from
bool bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& dout, const Tensor& lse, const OptTensor& delta, const Tensor& dq,
         const Tensor& dk, const Tensor& dv, double scale, int64_t row_begin, int64_t row_count, const OptTensor& kv_len,
         const OptTensor& kv_start, const OptTensor& kv_end, int64_t accumulate_dkv, const Tensor& ws, const OptTensor& bias,
         const OptTensor& o) {
    lvx_attn_shape s;
    if (!fill_shape(s, q, k, v, scale, kv_len, kv_start, kv_end) || !fill_bias(s, bias, q)) return false;
    const at::ScalarType kv_type = accumulate_dkv ? at::kFloat : q.scalar_type();
    if (!plain4(dout, q, q.scalar_type()) || dout.sizes() != q.sizes() || !rows_ok(lse, q) || !delta == !o ||
        (delta && !rows_ok(*delta, q)) || (o && (!plain4(*o, q, q.scalar_type()) || o->sizes() != q.sizes())) || !plain4(dq, q, q.scalar_type()) || dq.sizes() != q.sizes() || !plain4(dk, q, kv_type) || dk.sizes() != k.sizes() ||
        !plain4(dv, q, kv_type) || dv.sizes() != k.sizes())
        return false;
    const lvx_tensor tq = t4(q), tk = t4(k), tv = t4(v), td = t4(dout), tdq = t4(dq), tdk = t4(dk), tdv = t4(dv);
    const float *const lp = lse.data_ptr<float>(), *const dp = delta ? delta->data_ptr<float>() : nullptr;
    const lvx_tensor to = o ? t4(*o) : lvx_tensor{};
    void *const wp = ws.data_ptr(), *const st = current_stream();
    const size_t wb = ws.nbytes();
    call("lvx_bwd", [&] {
        if (o)
            return lib.bwd_from_o(&s, &tq, &tk, &tv, &to, &td, lp, &tdq, &tdk, &tdv, (int32_t)accumulate_dkv, (int32_t)row_begin,
                                  (int32_t)row_count, wp, wb, st);
        return lib.bwd(&s, &tq, &tk, &tv, &td, lp, dp, &tdq, &tdk, &tdv, (int32_t)accumulate_dkv, (int32_t)row_begin, (int32_t)row_count,
                       wp, wb, st);
    });
    return true;
}

// (kv_start, kv_end) of the hull of what a bias leaves visible, int32 [B, Lq] each, or None.
py::object bias_hull(const Tensor& q, const Tensor& k, const Tensor& bias) {
    lvx_attn_shape s;
    if (!fill_shape(s, q, k, k, 1.0, {}, {}, {}) || !fill_bias(s, bias, q)) return py::none();
    Tensor start = at::empty({s.B, s.Lq}, q.options().dtype(at::kInt)), end = at::empty({s.B, s.Lq}, q.options().dtype(at::kInt));
    int32_t *const sp = start.data_ptr<int32_t>(), *const ep = end.data_ptr<int32_t>();
    void* const st = current_stream();
    call("lvx_bias_hull", [&] { return lib.bias_hull(&s, sp, ep, st); });
    return py::make_tuple(std::move(start), std::move(end));
}

// Bytes of the backward's workspace for a window of `rows` rows, or -1.
int64_t bwd_workspace_bytes(const Tensor& q, const Tensor& k, int64_t rows, const OptTensor& kv_len, const OptTensor& kv_start,
                            const OptTensor& kv_end, bool accumulate_dkv) {
    lvx_attn_shape s;
    if (!fill_shape(s, q, k, k, 1.0, kv_len, kv_start, kv_end)) return -1;
    return (int64_t)(accumulate_dkv ? lib.bwd_acc_workspace_bytes : lib.bwd_workspace_bytes)(&s, (int32_t)rows);
}

// (dq, dk, dv) of a backward: dq contiguous, or in q's memory order with `like_q`; dk and dv views of
// [B, Lkv, Hkv, D] memory.
py::tuple backward_outputs(const Tensor& q, const Tensor& k, bool like_q) {
    Tensor dq = like_q ? at::empty_like(q) : at::empty(q.sizes(), q.options());
    const auto kv = [&] { return at::empty({k.size(0), k.size(2), k.size(1), k.size(3)}, q.options()).transpose(1, 2); };
    Tensor dk = kv(), dv = kv();
    return py::make_tuple(std::move(dq), std::move(dk), std::move(dv));
}

uintptr_t stream_of(int64_t device) {
    return reinterpret_cast<uintptr_t>(c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream());
}

}  // namespace

PYBIND11_MODULE(_lvx_host, m) {
    m.def("bind", &bind);
    m.def("usable", &usable);
    m.def("forward_buffers", &forward_buffers);
    m.def("round_buffers", &round_buffers);
    m.def("fwd", &fwd);
    m.def("bwd_preprocess", &bwd_preprocess);
    m.def("bwd", &bwd);
    m.def("bwd_workspace_bytes", &bwd_workspace_bytes);
    m.def("bias_hull", &bias_hull);
    m.def("backward_outputs", &backward_outputs);
    m.def("stream_of", &stream_of);
}

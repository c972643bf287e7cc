// The host side of the package's operations: checks, output allocation and launches, on torch tensors, for the Python
// layer above it and the torch.library ops' CUDA kernels.
//
// A small attention or a layer of the model is paced by its host work: in Python, a call's checks, allocations, ctypes
// conversions and stream look-ups took 10 to 15 us around a 5 us kernel, and a layer's products added a dispatch each.
// Here a call is one binding, and a layer's forward or backward is one function. Autograd stays in Python (the
// autograd.Functions hold the graph), and the kernels stay behind the C ABI in libnanonemo_fa.so, which this module
// links: nothing here launches a kernel of its own.
//
// Every function allocates through PyTorch's caching allocator, launches on PyTorch's current stream of its inputs'
// device, and neither synchronises nor keeps state between calls.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>
#include <torch/library.h>

#include <array>
#include <cmath>
#include <functional>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "nanonemo_fa.h"
#include "nanonemo_linear.h"
#include "nanonemo_loss.h"
#include "nanonemo_rmsnorm.h"
#include "nanonemo_rope.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using S3 = std::array<int64_t, 3>;
using T2 = std::tuple<Tensor, Tensor>;
using T3 = std::tuple<Tensor, Tensor, Tensor>;

[[noreturn]] void raise(const std::string& what) { throw std::runtime_error(what); }
void need(bool ok, const char* what) {
    if (!ok) raise(what);
}
void done(int rc, const char* (*last)()) {
    if (rc != 0) {
        const char* m = last();
        raise(m && *m ? m : "kernel library call failed with code " + std::to_string(rc));
    }
}
void fa_done(int rc) { done(rc, nn_fa_last_error); }
void rope_done(int rc) { done(rc, nn_rope_last_error); }
void rms_done(int rc) { done(rc, nn_rmsnorm_last_error); }
void lin_done(int rc) { done(rc, nn_linear_last_error); }
void loss_done(int rc) { done(rc, nn_loss_last_error); }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// The library's element type code: 0 fp16, 1 bf16, 2 fp32, -1 none of them.
int code(at::ScalarType t) { return t == at::kHalf ? 0 : t == at::kBFloat16 ? 1 : t == at::kFloat ? 2 : -1; }
int code(const Tensor& t) { return code(t.scalar_type()); }

// The tensor's values at its address: a gradient may come as a lazy negation of what lies there.
Tensor real_values(const Tensor& t) { return t.is_neg() ? t.resolve_neg() : t; }
Tensor contig(const Tensor& t) { return t.is_contiguous() && !t.is_neg() ? t : real_values(t).contiguous(); }
Tensor empty_of(const Tensor& like, at::IntArrayRef shape) { return at::empty(shape, like.options()); }
Tensor empty_f32(const Tensor& like, at::IntArrayRef shape) { return at::empty(shape, like.options().dtype(at::kFloat)); }
Tensor bytes(const Tensor& like, size_t n) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }
float scale_of(int64_t D) { return (float)(1.0 / std::sqrt((double)D)); }

// The library reads raw addresses on x's device.
void check_on_device(const Tensor& x, std::initializer_list<const Tensor*> others) {
    need(x.is_cuda(), "inputs must be CUDA tensors");
    for (const Tensor* t : others) need(t->device() == x.device(), "inputs must be CUDA tensors on the same device");
}

// ---- attention ----------------------------------------------------------------------------------

// The reference's check_inputs (flash_attn.cu:342-356) with the dtypes widened to {fp16, bf16}. seq is 2 for
// (B, heads, T, hd) tensors and 1 for (B, T, heads, hd).
void check_attention(const Tensor& q, const Tensor& k, const Tensor& v, int seq) {
    const int hd = 3 - seq;
    need(q.is_cuda() && k.is_cuda() && v.is_cuda(), "inputs must be CUDA tensors");
    const int c = code(q);
    need((c == 0 || c == 1) && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(),
         "inputs must be float16 or bfloat16 (all the same dtype)");
    need(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "expected (B, H, T, hd) / (B, KVH, T, hd)");
    need(q.size(0) == k.size(0) && q.size(seq) == k.size(seq) && k.sizes() == v.sizes(),
         "K and V must share shape; Q must share batch and length");
    need(q.size(3) == k.size(3), "Q and K must share head_dim");
    need(q.size(3) == 32 || q.size(3) == 64, "head_dim must be 32 or 64");
    need(k.size(hd) != 0 && q.size(hd) % k.size(hd) == 0, "query heads must group evenly over KV heads");
    need(q.device() == k.device() && q.device() == v.device(), "inputs must be on the same device");
    for (const Tensor* t : {&q, &k, &v})
        need(t->numel() == 0 || (uintptr_t)t->data_ptr() % 16 == 0, "inputs must be 16-byte aligned");
}

// The {batch, head, row} element strides through which the kernels can read the (B, heads, T, hd) tensor in place, if
// they can: unit hd stride, the others positive multiples of 8 elements (16-byte rows) with rows at least hd apart and
// within the library's 32-bit row offsets, and a 16-byte aligned start. A dimension of size 1 has no stride of its
// own; the dense one stands for it.
std::optional<S3> strides_of(const Tensor& t) {
    if (t.dim() != 4 || t.numel() == 0) return std::nullopt;
    const int64_t B = t.size(0), H = t.size(1), T = t.size(2), D = t.size(3);
    const int64_t st = T > 1 ? t.stride(2) : D, sh = H > 1 ? t.stride(1) : T * st, sb = B > 1 ? t.stride(0) : H * sh;
    if (t.stride(3) != 1 || st < D || st % 8 || sh <= 0 || sh % 8 || sb <= 0 || sb % 8) return std::nullopt;
    if (T * st >= (int64_t)1 << 30 || sb >= (int64_t)1 << 40 || sh * H >= (int64_t)1 << 40) return std::nullopt;
    if ((uintptr_t)t.data_ptr() % 16) return std::nullopt;
    return S3{sb, sh, st};
}
S3 dense_strides(const Tensor& t) { return {t.size(1) * t.size(2) * t.size(3), t.size(2) * t.size(3), t.size(3)}; }
S3 known_strides(const Tensor& t) { return t.is_contiguous() ? dense_strides(t) : *strides_of(t); }

// Makes the tensors contiguous unless they all are, or the library can read them in place through strides they share
// (as it takes k and v, and q and dO).
void make_readable(std::initializer_list<Tensor*> ts) {
    bool dense = true;
    for (Tensor* t : ts) {
        *t = real_values(*t);
        dense = dense && t->is_contiguous();
    }
    if (dense) return;
    std::optional<S3> first;
    bool ok = true;
    for (Tensor* t : ts) {
        const auto s = strides_of(*t);
        ok = ok && s && (!first || *first == *s);
        if (s) first = s;
    }
    if (!ok)
        for (Tensor* t : ts) *t = t->contiguous();
}

bool empty_problem(const Tensor& q) { return q.size(0) == 0 || q.size(1) == 0 || q.size(2) == 0; }

// (B, heads, T, hd): o and lse dense whatever the inputs' strides.
T2 fa_fwd(Tensor q, Tensor k, Tensor v) {
    make_readable({&q});
    make_readable({&k, &v});
    check_attention(q, k, v, 2);
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3), KVH = k.size(1);
    Tensor o = empty_of(q, q.sizes()), lse = empty_f32(q, {B, H, T});
    if (empty_problem(q)) return {o, lse};
    const c10::DeviceGuard guard(q.device());
    float* l = lse.data_ptr<float>();
    if (q.is_contiguous() && k.is_contiguous() && v.is_contiguous()) {
        fa_done(nn_fa_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, B, H, KVH, T, D, code(q), scale_of(D),
                          stream_of(q)));
    } else {
        const S3 s[3] = {known_strides(q), known_strides(k), dense_strides(o)};
        fa_done(nn_fa_fwd_views(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, B, H, KVH, T, D, s[0].data(), code(q),
                                scale_of(D), stream_of(q)));
    }
    return {o, lse};
}

// The backwards check what they are given like the forwards: a saved tensor is what the caller's saved-tensor hooks made
// of it, and the library reads raw addresses.
void check_backward(const Tensor& d_o, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, int seq) {
    check_attention(q, k, v, seq);
    check_on_device(q, {&d_o, &o, &lse});
    need(d_o.sizes() == q.sizes() && d_o.scalar_type() == q.scalar_type() && o.sizes() == q.sizes() && o.scalar_type() == q.scalar_type(),
         "d_o must be a contiguous float16/bfloat16 tensor shaped like q");
    need(lse.sizes() == at::IntArrayRef({q.size(0), q.size(3 - seq), q.size(seq)}) && lse.scalar_type() == at::kFloat,
         "lse must be a float32 tensor of shape (B, H, T)");
}

T3 fa_bwd(Tensor d_o, Tensor q, Tensor k, Tensor v, const Tensor& o_, const Tensor& lse_) {
    make_readable({&q, &d_o});
    make_readable({&k, &v});
    check_backward(d_o, q, k, v, o_, lse_, 2);
    const Tensor o = contig(o_), lse = contig(lse_);
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3), KVH = k.size(1);
    Tensor dq = empty_of(q, q.sizes()), dk = empty_of(k, k.sizes()), dv = empty_of(v, v.sizes());
    if (empty_problem(q)) return {dq, dk, dv};
    const c10::DeviceGuard guard(q.device());
    const size_t n = nn_fa_bwd_workspace_size(B, H, KVH, T, D);
    Tensor ws = bytes(q, n);
    const float* l = lse.data_ptr<float>();
    if (q.is_contiguous() && d_o.is_contiguous() && k.is_contiguous() && v.is_contiguous()) {
        fa_done(nn_fa_bwd(d_o.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, dq.data_ptr(), dk.data_ptr(),
                          dv.data_ptr(), ws.data_ptr(), n, B, H, KVH, T, D, code(q), scale_of(D), stream_of(q)));
    } else {
        const S3 s[5] = {known_strides(q), known_strides(k), dense_strides(o), dense_strides(dq), dense_strides(dk)};
        fa_done(nn_fa_bwd_views(d_o.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, dq.data_ptr(),
                                dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), n, B, H, KVH, T, D, s[0].data(), code(q),
                                scale_of(D), stream_of(q)));
    }
    return {dq, dk, dv};
}

S3 bthd_strides(const Tensor& t) { return {t.size(1) * t.size(2) * t.size(3), t.size(3), t.size(2) * t.size(3)}; }

// (B, T, heads, hd), contiguous copies where needed.
T2 bthd_fwd(const Tensor& q_, const Tensor& k_, const Tensor& v_) {
    const Tensor q = contig(q_), k = contig(k_), v = contig(v_);
    check_attention(q, k, v, 1);
    const int64_t B = q.size(0), T = q.size(1), H = q.size(2), D = q.size(3);
    Tensor o = empty_of(q, q.sizes()), lse = empty_f32(q, {B, H, T});
    if (empty_problem(q)) return {o, lse};
    const c10::DeviceGuard guard(q.device());
    fa_done(nn_fa_fwd_strided(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(), B, H, k.size(2), T, D,
                              bthd_strides(q).data(), bthd_strides(k).data(), code(q), scale_of(D), stream_of(q)));
    return {o, lse};
}

T3 bthd_bwd(const Tensor& d_o_, const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_, const Tensor& lse_) {
    const Tensor d_o = contig(d_o_), q = contig(q_), k = contig(k_), v = contig(v_), o = contig(o_), lse = contig(lse_);
    check_backward(d_o, q, k, v, o, lse, 1);
    const int64_t B = q.size(0), T = q.size(1), H = q.size(2), D = q.size(3), KVH = k.size(2);
    Tensor dq = empty_of(q, q.sizes()), dk = empty_of(k, k.sizes()), dv = empty_of(v, v.sizes());
    if (empty_problem(q)) return {dq, dk, dv};
    const c10::DeviceGuard guard(q.device());
    const size_t n = nn_fa_bwd_workspace_size(B, H, KVH, T, D);
    Tensor ws = bytes(q, n);
    fa_done(nn_fa_bwd_strided(d_o.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(),
                              dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), n, B, H, KVH, T, D,
                              bthd_strides(q).data(), bthd_strides(k).data(), code(q), scale_of(D), stream_of(q)));
    return {dq, dk, dv};
}

// The RoPE tables: float32 (T_max >= T, hd/2), on the inputs' GPU. Checked before any launch, since the library reads
// them through raw device pointers (a host table would be read as device memory).
void check_tables(const Tensor& cos, const Tensor& sin, int64_t T, int64_t D, c10::Device device) {
    need(cos.is_cuda() && sin.is_cuda() && cos.device() == device && sin.device() == device && cos.scalar_type() == at::kFloat &&
             sin.scalar_type() == at::kFloat && cos.sizes() == sin.sizes() && cos.dim() == 2 && cos.size(1) == D / 2 && cos.size(0) >= T,
         "cos/sin must be float32 (T_max >= T, hd/2) tables on the inputs' device");
}

// RoPE of q folded in: (o, lse, rotated q).
T3 bthd_rope_fwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& cos_, const Tensor& sin_) {
    const Tensor q = contig(q_), k = contig(k_), v = contig(v_);
    check_attention(q, k, v, 1);
    const int64_t B = q.size(0), T = q.size(1), H = q.size(2), D = q.size(3);
    check_tables(cos_, sin_, T, D, q.device());
    const Tensor cos = contig(cos_), sin = contig(sin_);
    Tensor o = empty_of(q, q.sizes()), q_rot = empty_of(q, q.sizes()), lse = empty_f32(q, {B, H, T});
    if (empty_problem(q)) return {o, lse, q_rot};
    const c10::DeviceGuard guard(q.device());
    fa_done(nn_fa_fwd_rope_strided(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(), q_rot.data_ptr(),
                                   cos.data_ptr<float>(), sin.data_ptr<float>(), cos.size(0), B, H, k.size(2), T, D,
                                   bthd_strides(q).data(), bthd_strides(k).data(), code(q), scale_of(D), stream_of(q)));
    return {o, lse, q_rot};
}

T3 bthd_rope_bwd(const Tensor& d_o_, const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_, const Tensor& lse_,
                 const Tensor& cos_, const Tensor& sin_) {
    const Tensor d_o = contig(d_o_), q = contig(q_), k = contig(k_), v = contig(v_), o = contig(o_), lse = contig(lse_);
    check_backward(d_o, q, k, v, o, lse, 1);
    check_tables(cos_, sin_, q.size(1), q.size(3), q.device());
    const Tensor cos = contig(cos_), sin = contig(sin_);
    const int64_t B = q.size(0), T = q.size(1), H = q.size(2), D = q.size(3), KVH = k.size(2);
    Tensor dq = empty_of(q, q.sizes()), dk = empty_of(k, k.sizes()), dv = empty_of(v, v.sizes());
    if (empty_problem(q)) return {dq, dk, dv};
    const c10::DeviceGuard guard(q.device());
    const size_t n = nn_fa_bwd_workspace_size(B, H, KVH, T, D);
    Tensor ws = bytes(q, n);
    fa_done(nn_fa_bwd_rope_strided(d_o.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(),
                                   dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), n, cos.data_ptr<float>(),
                                   sin.data_ptr<float>(), cos.size(0), B, H, KVH, T, D, bthd_strides(q).data(),
                                   bthd_strides(k).data(), code(q), scale_of(D), stream_of(q)));
    return {dq, dk, dv};
}

// The backward ops as the dispatcher calls them. A capture of the autograd engine's backward is refused (such a capture
// once ended in a host fault and no cause has been shown); capture without autograd is not affected.
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }
void refuse_capture_from_engine(const std::string& where, const std::function<bool()>& captures = capturing) {
    if (!torch::autograd::get_current_node() || !captures()) return;
    raise(where + ": capturing this op into a HIP graph while autograd records it (torch.cuda.graph around the "
          "forward and its autograd backward, or torch.compile(mode='reduce-overhead')) is not supported: such a capture once "
          "ended in a host fault in capture_end and no cause has been shown. Capture the C ABI calls (nn_fa_fwd / nn_fa_bwd / "
          "nn_fa_bwd_noalloc) instead, or run the ops eagerly (torch.compile(fullgraph=True) without graphs is supported).");
}
T3 fa_bwd_op(const Tensor& d_o, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse) {
    refuse_capture_from_engine("flash_attn backward op");
    return fa_bwd(d_o, q, k, v, o, lse);
}
T3 bthd_bwd_op(const Tensor& d_o, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse) {
    refuse_capture_from_engine("flash_attn_bthd backward op");
    return bthd_bwd(d_o, q, k, v, o, lse);
}
T3 bthd_rope_bwd_op(const Tensor& d_o, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse,
                    const Tensor& cos, const Tensor& sin) {
    refuse_capture_from_engine("flash_attn_bthd_rope backward op");
    return bthd_rope_bwd(d_o, q, k, v, o, lse, cos, sin);
}

// ---- RoPE ---------------------------------------------------------------------------------------

T2 rope(const Tensor& q_, const Tensor& k_, const Tensor& cos_, const Tensor& sin_, bool inverse) {
    check_on_device(q_, {&k_, &cos_, &sin_});
    need(q_.dim() == 4 && k_.dim() == 4 && q_.size(0) == k_.size(0) && q_.size(1) == k_.size(1) && q_.size(3) == k_.size(3),
         "expected q (B, T, H, hd) and k (B, T, KVH, hd)");
    need(code(q_) >= 0 && k_.scalar_type() == q_.scalar_type(), "q and k must share a dtype in {float16, bfloat16, float32}");
    const int64_t B = q_.size(0), T = q_.size(1), H = q_.size(2), KVH = k_.size(2), D = q_.size(3);
    need(D % 16 == 0, "head_dim must be a multiple of 16");
    need(cos_.scalar_type() == at::kFloat && sin_.scalar_type() == at::kFloat && cos_.sizes() == sin_.sizes() && cos_.dim() == 2 &&
             cos_.size(1) == D / 2 && cos_.size(0) >= T,
         "cos/sin must be float32 (T_max >= T, hd/2) tables");
    const Tensor q = contig(q_), k = contig(k_), cos = contig(cos_), sin = contig(sin_);
    Tensor qo = empty_of(q, q.sizes()), ko = empty_of(k, k.sizes());
    if (q.numel() == 0 && k.numel() == 0) return {qo, ko};
    const c10::DeviceGuard guard(q.device());
    const S3 qs{T * H * D, H * D, D}, ks{T * KVH * D, KVH * D, D};
    rope_done((inverse ? nn_rope_qk_bwd : nn_rope_qk)(q.data_ptr(), qo.data_ptr(), k.data_ptr(), ko.data_ptr(), cos.data_ptr<float>(),
                                                      sin.data_ptr<float>(), B, T, H, KVH, D, qs.data(), ks.data(), cos.size(0),
                                                      code(q), stream_of(q)));
    return {qo, ko};
}
T2 rope_op(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin) { return rope(q, k, cos, sin, false); }
T2 rope_bwd_op(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin) { return rope(q, k, cos, sin, true); }

// ---- residual add + RMSNorm ---------------------------------------------------------------------

int norm_code(at::ScalarType t) {
    const int c = code(t);
    if (c < 0) raise(std::string("only float32, float16 and bfloat16 are supported, got ") + c10::toString(t));
    return c;
}

T3 norm_fwd(const Tensor& x_, const OptTensor& delta_, const Tensor& weight_, double eps, at::ScalarType out_dtype) {
    need(x_.is_cuda(), "x must be a CUDA tensor");
    const bool has = delta_.has_value();
    check_on_device(x_, {&weight_, has ? &*delta_ : &x_});
    const Tensor x = contig(x_), w = contig(weight_), delta = has ? contig(*delta_) : Tensor();
    need(w.scalar_type() == at::kFloat, "weight must be contiguous float32");
    if (has) need(delta.sizes() == x.sizes(), "delta must match x");
    const int64_t N = x.size(-1);
    need(w.numel() == N, "weight must have hidden-size elements");
    const int64_t M = N ? x.numel() / N : 0;
    Tensor y = at::empty(x.sizes(), x.options().dtype(out_dtype));
    Tensor h = has ? at::empty(x.sizes(), x.options().dtype(c10::promoteTypes(x.scalar_type(), delta.scalar_type()))) : empty_of(x, {0});
    Tensor rstd = empty_f32(x, x.sizes().slice(0, x.dim() - 1));
    const c10::DeviceGuard guard(x.device());
    rms_done(nn_add_rmsnorm_fwd(x.data_ptr(), has ? delta.data_ptr() : nullptr, w.data_ptr<float>(), y.data_ptr(),
                                has ? h.data_ptr() : nullptr, rstd.data_ptr<float>(), M, N, (float)eps, norm_code(x.scalar_type()),
                                has ? norm_code(delta.scalar_type()) : 0, norm_code(out_dtype), stream_of(x)));
    return {y, h, rstd};
}

T3 norm_bwd(const Tensor& dy_, const OptTensor& dh_, const Tensor& h_, const Tensor& weight_, const Tensor& rstd_,
            at::ScalarType dx_dtype, std::optional<at::ScalarType> ddelta_dtype) {
    const bool has = dh_.has_value();
    check_on_device(h_, {&dy_, &weight_, &rstd_, has ? &*dh_ : &h_});
    const Tensor dy = contig(dy_), h = contig(h_), w = contig(weight_), rstd = contig(rstd_), dh = has ? contig(*dh_) : Tensor();
    need(dy.sizes() == h.sizes(), "dy and h must be contiguous, same shape");
    need(has == ddelta_dtype.has_value(), "dh and ddelta_dtype go together");
    if (has) need(dh.scalar_type() == h.scalar_type(), "dh must be contiguous, h's dtype");
    const int64_t N = h.size(-1), M = N ? h.numel() / N : 0;
    need(w.numel() == N && (N == 0 || rstd.numel() == M), "weight must have hidden-size elements and rstd one per row");
    Tensor dx = at::empty(h.sizes(), h.options().dtype(dx_dtype));
    Tensor dd = has ? at::empty(h.sizes(), h.options().dtype(*ddelta_dtype)) : empty_of(h, {0});
    Tensor dw = empty_f32(h, {N});
    const size_t n = nn_add_rmsnorm_bwd_workspace_size(M, N);
    Tensor ws = bytes(h, n ? n : 1);
    const c10::DeviceGuard guard(h.device());
    rms_done(nn_add_rmsnorm_bwd(dy.data_ptr(), has ? dh.data_ptr() : nullptr, h.data_ptr(), w.data_ptr<float>(), rstd.data_ptr<float>(),
                                dx.data_ptr(), has ? dd.data_ptr() : nullptr, dw.data_ptr<float>(), ws.data_ptr(), n, M, N,
                                norm_code(dy.scalar_type()), norm_code(h.scalar_type()), norm_code(dx_dtype),
                                has ? norm_code(*ddelta_dtype) : 0, stream_of(h)));
    return {dx, dd, dw.to(w.scalar_type())};
}

// ---- linear layers ------------------------------------------------------------------------------
// The layers below run inside autograd.Functions, on flat (tokens, features) tensors of one 16-bit type: their
// products skip the autograd and autocast keys.
struct Inner {
    at::AutoDispatchBelowADInplaceOrView below;
    c10::impl::ExcludeDispatchKeyGuard no_autocast{c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA)};
};

// A tensor that the forward saved, as the kernels read it (see check_backward).
Tensor saved(const Tensor& t, const Tensor& x, at::IntArrayRef sizes, at::ScalarType type) {
    need(t.device() == x.device() && t.scalar_type() == type && t.sizes() == sizes,
         "a saved tensor is not what the forward saved: another device, type or shape");
    return contig(t);
}
Tensor saved(const Tensor& t, const Tensor& x, at::IntArrayRef sizes) { return saved(t, x, sizes, x.scalar_type()); }

// Above this many elements of dW the library's product fills the chip by itself and is the faster one (2048 x 2048 over
// 16384 tokens 140 us in this build's kernel against 165 with the cast, 4096 x 4096 over 8192 334 against 245); odd
// row counts are its too.
constexpr int64_t kWgradMost = 6000000;
// Whether dW (N, K) over T rows is the kernel's; so are only row counts within its 32-bit index.
bool wgrad_takes(int64_t T, int64_t N, int64_t K) { return N * K <= kWgradMost && N % 8 == 0 && T < (int64_t)1 << 30; }

// The tensor as the kernel reads it: rows of unit stride within its 32-bit offsets, 16-byte aligned (a gradient may
// arrive as a slice of anything).
Tensor rows_aligned(const Tensor& t) {
    const bool ok = t.stride(1) == 1 && t.stride(0) % 8 == 0 && t.stride(0) >= t.size(1) && t.stride(0) < (1 << 23) &&
                    (uintptr_t)t.data_ptr() % 16 == 0;
    return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

std::vector<Tensor> wgrad(const Tensor& dy_, const Tensor& x_, const std::vector<int64_t>& rows) {
    check_on_device(x_, {&dy_});
    need(dy_.dim() == 2 && x_.dim() == 2 && dy_.size(0) == x_.size(0) && dy_.scalar_type() == x_.scalar_type() && code(x_) >= 0 && code(x_) < 2,
         "expected float16 or bfloat16 gradients (T, N) and inputs (T, K)");
    const int64_t T = dy_.size(0), N = dy_.size(1), K = x_.size(1);
    const c10::DeviceGuard guard(x_.device());
    if (!wgrad_takes(T, N, K)) {
        // (dense rows are the library's to read whatever their width; an odd vocabulary's are not 16-byte aligned)
        auto dense = [](const Tensor& t) { return t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0 ? t : rows_aligned(t); };
        Tensor dw = at::mm(dense(dy_).t(), dense(x_), at::kFloat);
        if (rows.size() == 1) return {dw};
        std::vector<Tensor> out = dw.split_with_sizes(rows);
        for (Tensor& t : out) t = t.clone();
        return out;
    }
    const Tensor dy = rows_aligned(dy_), x = rows_aligned(x_);
    std::vector<Tensor> out;
    std::vector<float*> p;
    for (int64_t r : rows) {
        out.push_back(empty_f32(x, {r, K}));
        p.push_back(out.back().data_ptr<float>());
    }
    const size_t n = nn_linear_wgrad_workspace_size(T, N, K);
    Tensor ws = n ? bytes(x, n) : Tensor();
    lin_done(nn_linear_wgrad(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), T, N, K, (int)rows.size(), p.data(), rows.data(),
                             n ? ws.data_ptr() : nullptr, n, code(x), stream_of(x)));
    return out;
}

// Each group of fp32 (N_i, K) weights stacked into one (sum N_i, K) 16-bit tensor, in one launch: for the layers'
// products, and for the products of their inputs' gradients (the same tensors, or, `turned`, transposed copies, seen as
// (sum N_i, K), which the library multiplies by faster; every N_i is then a multiple of 8).
struct Weights {
    std::vector<Tensor> fwd, bwd;
};
Weights cast_weights(const Tensor& like, const std::vector<std::vector<Tensor>>& groups, bool turned) {
    Weights out;
    std::vector<const float*> src;
    std::vector<void*> dst, dst_t;
    std::vector<int64_t> count, rows, cols, ldt;
    for (const auto& g : groups) {
        int64_t N = 0;
        const int64_t K = g[0].size(1);
        for (const Tensor& w : g) {
            check_on_device(like, {&w});
            need(w.dim() == 2 && w.size(1) == K && w.is_contiguous(), "weights must be contiguous and of one width");
            N += w.size(0);
        }
        out.fwd.push_back(empty_of(like, {N, K}));
        const Tensor t = turned ? empty_of(like, {K, N}) : Tensor();
        out.bwd.push_back(turned ? t.t() : out.fwd.back());
        char *at = (char*)out.fwd.back().data_ptr(), *at_t = turned ? (char*)t.data_ptr() : nullptr;
        for (const Tensor& w : g) {
            src.push_back(w.data_ptr<float>());
            dst.push_back(at);
            count.push_back(w.numel());
            at += 2 * w.numel();
            if (!turned) continue;
            dst_t.push_back(at_t);
            at_t += 2 * w.size(0);
            rows.push_back(w.size(0)), cols.push_back(K), ldt.push_back(N);
        }
    }
    const int n = (int)src.size(), dt = code(like);
    lin_done(turned ? nn_linear_cast_both(n, src.data(), dst.data(), dst_t.data(), rows.data(), cols.data(), ldt.data(), dt, stream_of(like))
                    : nn_linear_cast(n, src.data(), dst.data(), count.data(), dt, stream_of(like)));
    return out;
}

// Layers that share an input: (their outputs side by side, the stacked 16-bit weights for the backward).
T2 project_fwd(const Tensor& x, const std::vector<Tensor>& ws, bool turned) {
    const Inner inner;
    const c10::DeviceGuard guard(x.device());
    const Weights w = cast_weights(x, {ws}, turned);
    return {at::mm(x, w.fwd[0].t()), w.bwd[0]};
}

// The attention layer (kernels/hip/layers.py): sizes, and the strides of its tensors for the library. q, k and v are
// column ranges of one (B T, n) product, dq, dk and dv of another such buffer.
struct LayerShape {
    int64_t B, T, H, KVH, D, nq, nk, n;
    int64_t fwd[9], bwd[15], rot[12], unrot[12];
    LayerShape(int64_t B, int64_t T, int64_t H, int64_t KVH, int64_t D) : B(B), T(T), H(H), KVH(KVH), D(D) {
        nq = H * D, nk = KVH * D, n = nq + 2 * nk;
        const S3 dense{T * nq, D, nq}, wide{T * n, D, n};            // {batch, head, row}
        const S3 dense_r{T * nq, nq, D}, wide_r{T * n, n, D};        // {batch, position, head}
        auto put = [](int64_t* to, std::initializer_list<S3> all) {
            for (const S3& s : all)
                for (int64_t v : s) *to++ = v;
        };
        put(fwd, {dense, wide, dense});                              // q, k and v, o
        put(bwd, {dense, wide, dense, wide, wide});                  // q and dO, k and v, o, dq, dk and dv
        put(rot, {wide_r, dense_r, wide_r, wide_r});                 // q out of the buffer, k in place
        put(unrot, {wide_r, wide_r, wide_r, wide_r});
    }
    char* k(const Tensor& buf) const { return (char*)buf.data_ptr() + 2 * nq; }
    char* v(const Tensor& buf) const { return k(buf) + 2 * nk; }
};

std::vector<Tensor> attention_layer_fwd(const Tensor& x, const Tensor& cos, const Tensor& sin, int64_t B, int64_t T, int64_t H,
                                        int64_t KVH, const Tensor& wq, const Tensor& wk, const Tensor& wv, const Tensor& wo,
                                        bool turned) {
    const Inner inner;
    const c10::DeviceGuard guard(x.device());
    const LayerShape s(B, T, H, KVH, wq.size(0) / H);
    check_tables(cos, sin, T, s.D, x.device());
    const int dt = code(x);
    void* st = stream_of(x);
    const Weights w = cast_weights(x, {{wq, wk, wv}, {wo}}, turned);
    Tensor qkv = at::mm(x, w.fwd[0].t());
    Tensor q = empty_of(x, {B * T, s.nq}), o = empty_of(x, {B * T, s.nq}), lse = empty_f32(x, {B, H, T});
    rope_done(nn_rope_qk_views(qkv.data_ptr(), q.data_ptr(), s.k(qkv), s.k(qkv), cos.data_ptr<float>(), sin.data_ptr<float>(), B, T, H,
                               KVH, s.D, s.rot, cos.size(0), dt, 0, st));
    fa_done(nn_fa_fwd_views(q.data_ptr(), s.k(qkv), s.v(qkv), o.data_ptr(), lse.data_ptr<float>(), B, H, KVH, T, s.D, s.fwd, dt,
                            scale_of(s.D), st));
    return {at::mm(o, w.fwd[1].t()), qkv, q, o, lse, w.bwd[0], w.bwd[1]};
}

// The gradients of x, wq, wk, wv and wo; undefined where not needed.
std::vector<OptTensor> attention_layer_bwd(const Tensor& dy_, const Tensor& x, const Tensor& cos_, const Tensor& sin_, const Tensor& qkv_,
                                           const Tensor& q_, const Tensor& o_, const Tensor& lse_, const Tensor& w, const Tensor& wo,
                                           int64_t B, int64_t T, int64_t H, int64_t KVH, bool need_x, bool need_qkv, bool need_o) {
    const Inner inner;
    check_on_device(x, {&dy_});
    const c10::DeviceGuard guard(x.device());
    const LayerShape s(B, T, H, KVH, wo.size(1) / H);
    check_tables(cos_, sin_, T, s.D, x.device());
    const Tensor cos = contig(cos_), sin = contig(sin_), lse = saved(lse_, x, {B, H, T}, at::kFloat);
    const Tensor qkv = saved(qkv_, x, {B * T, s.n}), q = saved(q_, x, {B * T, s.nq}), o = saved(o_, x, {B * T, s.nq});
    const int dt = code(x);
    void* st = stream_of(x);
    const Tensor dy = contig(dy_);
    std::vector<OptTensor> out(5);
    Tensor d_o = need_x || need_qkv ? at::mm(dy, wo) : Tensor();
    if (need_o) out[4] = wgrad(dy, o, {wo.size(0)})[0];
    if (!need_x && !need_qkv) return out;
    Tensor dqkv = at::empty_like(qkv);
    const size_t n = nn_fa_bwd_workspace_size(B, H, KVH, T, s.D);
    Tensor ws = bytes(x, n);
    fa_done(nn_fa_bwd_views(d_o.data_ptr(), q.data_ptr(), s.k(qkv), s.v(qkv), o.data_ptr(), lse.data_ptr<float>(), dqkv.data_ptr(),
                            s.k(dqkv), s.v(dqkv), ws.data_ptr(), n, B, H, KVH, T, s.D, s.bwd, dt, scale_of(s.D), st));
    rope_done(nn_rope_qk_views(dqkv.data_ptr(), dqkv.data_ptr(), s.k(dqkv), s.k(dqkv), cos.data_ptr<float>(), sin.data_ptr<float>(), B, T,
                               H, KVH, s.D, s.unrot, cos.size(0), dt, 1, st));
    if (need_x) out[0] = at::mm(dqkv, w);
    if (need_qkv) {
        auto dw = wgrad(dqkv, x, {s.nq, s.nk, s.nk});
        for (int i = 0; i < 3; ++i) out[1 + i] = dw[i];
    }
    return out;
}

std::vector<Tensor> mlp_fwd(const Tensor& x, const Tensor& w_gate, const Tensor& w_up, const Tensor& w_down, bool turned) {
    const Inner inner;
    const c10::DeviceGuard guard(x.device());
    const Weights w = cast_weights(x, {{w_gate, w_up}, {w_down}}, turned);
    Tensor gu = at::mm(x, w.fwd[0].t());
    const int64_t T = x.size(0), F = w_gate.size(0);
    Tensor h = empty_of(x, {T, F});
    lin_done(nn_swiglu_fwd(gu.data_ptr(), h.data_ptr(), T, F, code(x), stream_of(x)));
    return {at::mm(h, w.fwd[1].t()), gu, h, w.bwd[0], w.bwd[1]};
}

// The gradients of x, w_gate, w_up and w_down; undefined where not needed.
std::vector<OptTensor> mlp_bwd(const Tensor& dy_, const Tensor& x, const Tensor& gu_, const Tensor& h_, const Tensor& w, const Tensor& w_down,
                               bool need_x, bool need_gu, bool need_down) {
    const Inner inner;
    check_on_device(x, {&dy_});
    const c10::DeviceGuard guard(x.device());
    const int64_t T = x.size(0), F = w_down.size(1);
    const Tensor dy = contig(dy_), gu = saved(gu_, x, {T, 2 * F}), h = saved(h_, x, {T, F});
    std::vector<OptTensor> out(4);
    Tensor dh = need_x || need_gu ? at::mm(dy, w_down) : Tensor();
    if (need_down) out[3] = wgrad(dy, h, {w_down.size(0)})[0];
    if (!need_x && !need_gu) return out;
    Tensor dgu = at::empty_like(gu);
    lin_done(nn_swiglu_bwd(dh.data_ptr(), gu.data_ptr(), dgu.data_ptr(), T, F, code(x), stream_of(x)));
    if (need_x) out[0] = at::mm(dgu, w);
    if (need_gu) {
        auto dw = wgrad(dgu, x, {F, F});
        out[1] = dw[0], out[2] = dw[1];
    }
    return out;
}

// (logits, loss, w16 for the backward, lse, 1 / rows that count).
std::vector<Tensor> head_fwd(const Tensor& x, const Tensor& w_, const Tensor& targets, bool turned) {
    const Inner inner;
    check_on_device(x, {&targets});
    need(targets.is_contiguous() && targets.numel() == x.size(0), "expected one contiguous target per row");
    const c10::DeviceGuard guard(x.device());
    const Weights w = cast_weights(x, {{w_}}, turned && w_.size(0) % 8 == 0);
    const Tensor logits = at::mm(x, w.fwd[0].t());
    const int64_t R = logits.size(0), V = logits.size(1);
    Tensor lse = empty_f32(x, {R}), rows = empty_f32(x, {R}), loss = empty_f32(x, {}), inv = empty_f32(x, {});
    loss_done(nn_cross_entropy_fwd(logits.data_ptr(), targets.data_ptr<int64_t>(), lse.data_ptr<float>(), rows.data_ptr<float>(),
                                   loss.data_ptr<float>(), inv.data_ptr<float>(), R, V, code(x), stream_of(x)));
    return {logits, loss, w.bwd[0], lse, inv};
}

// The gradients of x and w from those of the logits and of the loss (either may be missing); logits: the forward's, or
// nothing to compute them again (by the forward's product, on rows).
std::vector<OptTensor> head_bwd(const OptTensor& dlogits_, const OptTensor& dloss, const OptTensor& logits_, const Tensor& x,
                                const Tensor& w, const Tensor& targets_, const Tensor& lse_, const Tensor& inv_, bool need_x, bool need_w) {
    const Inner inner;
    check_on_device(x, {});
    const c10::DeviceGuard guard(x.device());
    const int64_t R = x.size(0), V = w.size(0);
    std::vector<OptTensor> out(2);
    Tensor d = dlogits_.has_value() ? saved(*dlogits_, x, {R, V}) : Tensor();
    if (dloss.has_value()) {
        const Tensor targets = saved(targets_, x, {R}, at::kLong), lse = saved(lse_, x, {R}, at::kFloat), inv = saved(inv_, x, {}, at::kFloat);
        const Tensor logits = logits_.has_value() ? saved(*logits_, x, {R, V}) : at::mm(x, contig(w).t()), g = saved(*dloss, x, {}, at::kFloat);
        Tensor t = at::empty_like(logits);
        loss_done(nn_cross_entropy_bwd(logits.data_ptr(), targets.data_ptr<int64_t>(), lse.data_ptr<float>(), inv.data_ptr<float>(),
                                       g.data_ptr<float>(), t.data_ptr(), R, V, code(x), stream_of(x)));
        d = d.defined() ? t.add_(d) : t;
    }
    if (!d.defined()) return out;
    if (need_x) out[0] = at::mm(d, w);
    if (need_w) out[1] = wgrad(d, x, {V})[0];
    return out;
}

// ---- routing ------------------------------------------------------------------------------------

// Whether the tensor's values lie at its address, as dense values of its own type: not inside a transform's wrapper
// (vmap, is_grads_batched, torch.func.grad, functionalization), not a lazy zero, negation or conjugate, not sparse,
// nested or a subclass with its own dispatch.
bool ordinary(const Tensor& t) {
    using K = c10::DispatchKey;
    static constexpr c10::DispatchKeySet wrapped({K::Python, K::Batched, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Functionalize,
                                                  K::ZeroTensor, K::Negative, K::Conjugate});
    return !t.key_set().has_any(wrapped) && !t.is_nested() && t.layout() == at::kStrided;
}
bool ordinary_py(const py::args& ts) {
    for (py::handle t : ts)
        if (!ordinary(THPVariable_Unpack(t.ptr()))) return false;
    return true;
}

// Whether every argument is a plain (ordinary, no subclass) CUDA tensor and neither a torch.func transform nor a Python dispatch mode is
// active (see kernels/hip/__init__.py, eager).
bool plain_cuda(const py::args& ts) {
    for (py::handle t : ts)
        if (!THPVariable_CheckExact(t.ptr()) || !THPVariable_Unpack(t.ptr()).is_cuda() || !ordinary(THPVariable_Unpack(t.ptr())))
            return false;
    // (a torch.func transform puts its key into the thread's set while its stack is not empty)
    return c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

py::object strides_py(const Tensor& t) {
    const auto s = strides_of(t);
    if (!s) return py::none();
    return py::make_tuple((*s)[0], (*s)[1], (*s)[2]);
}
std::vector<Tensor> readable_py(Tensor a, std::optional<Tensor> b) {
    if (!b) {
        make_readable({&a});
        return {a};
    }
    Tensor t = *b;
    make_readable({&a, &t});
    return {a, t};
}

}  // namespace

// The CUDA kernels of the torch.library ops, whose schemas, fake impls and autograd the Python modules register.
TORCH_LIBRARY_IMPL(nanonemo, CUDA, m) {
    m.impl("flash_attn", [](const Tensor& q, const Tensor& k, const Tensor& v) { return fa_fwd(q, k, v); });
    m.impl("flash_attn_bwd", fa_bwd_op);
    m.impl("flash_attn_bthd", bthd_fwd);
    m.impl("flash_attn_bthd_bwd", bthd_bwd_op);
    m.impl("flash_attn_bthd_rope", bthd_rope_fwd);
    m.impl("flash_attn_bthd_rope_bwd", bthd_rope_bwd_op);
    m.impl("rope_qk", rope_op);
    m.impl("rope_qk_bwd", rope_bwd_op);
    m.impl("cuda_add_rms_norm_fwd", norm_fwd);
    m.impl("cuda_add_rms_norm_bwd", norm_bwd);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    const auto nogil = py::call_guard<py::gil_scoped_release>();
    m.def("fa_fwd", fa_fwd, nogil);
    m.def("fa_bwd", fa_bwd, nogil);
    m.def("fa_bwd_op", fa_bwd_op, nogil);
    m.def("bthd_fwd", bthd_fwd, nogil);
    m.def("bthd_bwd", bthd_bwd, nogil);
    m.def("bthd_bwd_op", bthd_bwd_op, nogil);
    m.def("bthd_rope_fwd", bthd_rope_fwd, nogil);
    m.def("bthd_rope_bwd", bthd_rope_bwd, nogil);
    m.def("bthd_rope_bwd_op", bthd_rope_bwd_op, nogil);
    m.def("rope", rope, nogil);
    m.def("norm_fwd", norm_fwd, nogil);
    m.def("norm_bwd", norm_bwd, nogil);
    m.def("wgrad", wgrad, nogil);
    m.def("wgrad_takes", wgrad_takes);
    m.def("rows_aligned", rows_aligned);
    m.def("project_fwd", project_fwd, nogil);
    m.def("attention_layer_fwd", attention_layer_fwd, nogil);
    m.def("attention_layer_bwd", attention_layer_bwd, nogil);
    m.def("mlp_fwd", mlp_fwd, nogil);
    m.def("mlp_bwd", mlp_bwd, nogil);
    m.def("head_fwd", head_fwd, nogil);
    m.def("head_bwd", head_bwd, nogil);
    m.def("plain_cuda", plain_cuda);
    m.def("ordinary", ordinary_py);
    // A tensor's version counter (which its changes in place raise), without the tensor.
    py::class_<c10::VariableVersion>(m, "Version")
        .def(py::init([](const Tensor& t) { return t.unsafeGetTensorImpl()->version_counter(); }))
        .def("current", &c10::VariableVersion::current_version);
    m.def("check_tables", check_tables);
    m.def("refuse_capture_from_engine", [](const std::string& where, bool captures) {
        refuse_capture_from_engine(where, [captures] { return captures; });
    });
    m.def("strides_of", strides_py);
    m.def("readable", readable_py, py::arg("a"), py::arg("b") = std::nullopt);
}

// Compiled torch binding over the C ABI of libspear_btp.so: the module that stands where the
// reference has its extension module `spear._btp` (csrc/btp/_bindings.cu:240-243, built by
// CMakeLists.txt:86-101 there). It exports
//     forward (coeff, x, y, checkpoint, k, wpb)
//     backward(coeff, x, dy, checkpoint, dx, dA, k, wpb)
// with the reference's positional arguments, in-place semantics (the caller allocates every output)
// and argument checks and messages (csrc/btp/_bindings.cu:19-60, raised as RuntimeError by
// TORCH_CHECK), plus the shape / stride / device checks the reference leaves out, and the bindings
// of the entry points the reference has no counterpart for (log-space gates, fused layer layout).
// No kernel code lives here: every function unpacks tensors into raw pointers and sizes and calls
// the C ABI on torch's current stream of the tensors' device, without synchronising.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/extension.h>

#include <string>
#include <vector>

#include "../../include/spear_btp.h"
#include "../../include/spear_layer.h"

namespace {

int tag_of(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return SPEAR_BTP_BF16;
    case at::kHalf: return SPEAR_BTP_F16;
    case at::kFloat: return SPEAR_BTP_F32;
    default: return -1;
  }
}

bool is_16bit(const at::Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }

void check_layout(const char* name, const at::Tensor& t, at::IntArrayRef shape) {
  // The reference reads B*H*L (resp. B*H*16*L) elements without looking at shapes or strides
  // (csrc/btp/_bindings.cu:80-87); a wrong shape there is an out-of-bounds read. Here it raises.
  TORCH_CHECK(t.sizes() == shape, name, " must have shape ", shape, ", got ", t.sizes(), ".");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous.");
}

void check_same_device(std::initializer_list<const at::Tensor*> ts) {
  const at::Tensor* first = nullptr;
  for (const at::Tensor* t : ts) {
    if (t == nullptr || !t->defined()) continue;
    if (first == nullptr) first = t;
    TORCH_CHECK(t->device() == first->device(), "All tensors must be on the same device.");
  }
}

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void raise_native(int rc) {
  const char* msg = spear_btp_last_error();
  TORCH_CHECK(false, (msg && msg[0]) ? std::string(msg) : "spear_btp call failed with code " + std::to_string(rc));
}

void check_common(const at::Tensor& x, const at::Tensor& coeff, int64_t k, int64_t wpb, const char* wpb_msg) {
  TORCH_CHECK(x.dim() == 4, "x must be [B, H, 16, L].");
  TORCH_CHECK(x.size(2) == 16, "Channel dim (DH) must be 16.");
  TORCH_CHECK(k == 1 || k == 2, "k must be 1 or 2.");
  TORCH_CHECK(wpb == 4 || wpb == 8 || wpb == 16 || wpb == 32, wpb_msg, wpb);
  TORCH_CHECK(is_16bit(coeff), "coeff must be float16 or bfloat16.");
  TORCH_CHECK(x.scalar_type() == coeff.scalar_type(), "x dtype must match coeff.");
}

// csrc/btp/_bindings.cu:76-150. `flags` is an extension (default: store the carry checkpoint, as the
// reference does); without SPEAR_BTP_WRITE_CHECKPOINT the checkpoint may be a zero-element placeholder.
void forward(const at::Tensor& coeff, const at::Tensor& x, at::Tensor y, at::Tensor checkpoint, int64_t k,
             int64_t wpb, int64_t flags) {
  TORCH_CHECK(coeff.is_cuda() && x.is_cuda() && y.is_cuda() && checkpoint.is_cuda(), "All tensors must be CUDA.");
  check_common(x, coeff, k, wpb, "Unsupported WPB value: ");
  TORCH_CHECK(y.scalar_type() == at::kFloat || y.scalar_type() == x.scalar_type(), "y must be float32 or match x dtype.");
  TORCH_CHECK(checkpoint.scalar_type() == at::kFloat, "checkpoint must be float32.");
  const int64_t B = x.size(0), H = x.size(1), L = x.size(3);
  TORCH_CHECK(L % 16 == 0, "Length L must be multiple of 16");
  check_layout("coeff", coeff, {B, H, L});
  check_layout("x", x, {B, H, 16, L});
  check_layout("y", y, {B, H, 16, L});
  if ((flags & SPEAR_BTP_WRITE_CHECKPOINT) || checkpoint.numel() != 0) check_layout("checkpoint", checkpoint, {B, H, L / 16, 16});
  check_same_device({&coeff, &x, &y, &checkpoint});
  const c10::DeviceGuard guard(x.device());
  const int rc = spear_btp_forward(coeff.data_ptr(), x.data_ptr(), y.data_ptr(), static_cast<float*>(checkpoint.data_ptr()),
                                   (int)B, (int)H, (int)L, (int)k, tag_of(x.scalar_type()), tag_of(y.scalar_type()),
                                   (unsigned)flags, stream_of(x));
  if (rc != 0) raise_native(rc);
}

// csrc/btp/_bindings.cu:152-229. Every element of dA is written (it need not arrive zero-filled); the
// checkpoint is accepted for signature compatibility and not read. With SPEAR_BTP_DX_F32 in `flags`
// (an extension) dx is float32 and receives the kernel's fp32 values unrounded.
void backward(const at::Tensor& coeff, const at::Tensor& x, const at::Tensor& dy, const at::Tensor& checkpoint,
              at::Tensor dx, at::Tensor dA, int64_t k, int64_t wpb, int64_t flags) {
  TORCH_CHECK(coeff.is_cuda() && x.is_cuda() && dy.is_cuda() && checkpoint.is_cuda(), "coeff, x, dy, checkpoint must be CUDA.");
  TORCH_CHECK(dx.is_cuda() && dA.is_cuda(), "dx and dA must be CUDA.");
  check_common(x, coeff, k, wpb, "Unsupported WPB value for backward: ");
  if (flags & SPEAR_BTP_DX_F32) {
    TORCH_CHECK(dx.scalar_type() == at::kFloat, "dx must be float32 in the fp32 check mode.");
  } else {
    TORCH_CHECK(dx.scalar_type() == x.scalar_type(), "dx dtype must match x.");
  }
  if (flags & SPEAR_BTP_DA_16) {
    TORCH_CHECK(dA.scalar_type() == coeff.scalar_type(), "dA must match coeff dtype.");
  } else {
    TORCH_CHECK(dA.scalar_type() == at::kFloat, "dA must be float32.");
  }
  TORCH_CHECK(dy.scalar_type() == at::kFloat || dy.scalar_type() == x.scalar_type(), "dy must be float32 or match x dtype.");
  const int64_t B = x.size(0), H = x.size(1), L = x.size(3);
  TORCH_CHECK(L % 16 == 0, "Length L must be multiple of 16");
  check_layout("coeff", coeff, {B, H, L});
  check_layout("x", x, {B, H, 16, L});
  check_layout("dy", dy, {B, H, 16, L});
  check_layout("dx", dx, {B, H, 16, L});
  check_layout("dA", dA, {B, H, L});
  check_same_device({&coeff, &x, &dy, &dx, &dA});
  const c10::DeviceGuard guard(x.device());
  const int rc = spear_btp_backward(coeff.data_ptr(), x.data_ptr(), dy.data_ptr(),
                                    checkpoint.numel() ? static_cast<const float*>(checkpoint.data_ptr()) : nullptr,
                                    dx.data_ptr(), dA.data_ptr(), (int)B, (int)H, (int)L, (int)k,
                                    tag_of(x.scalar_type()), tag_of(dy.scalar_type()), (unsigned)flags, stream_of(x));
  if (rc != 0) raise_native(rc);
}

void check_log_common(const at::Tensor& gate, const at::Tensor& x, int64_t k) {
  TORCH_CHECK(gate.is_cuda() && x.is_cuda(), "All tensors must be CUDA.");
  TORCH_CHECK(x.dim() == 4, "x must be [B, H, 16, L].");
  TORCH_CHECK(x.size(2) == 16, "Channel dim (DH) must be 16.");
  TORCH_CHECK(k == 1 || k == 2, "k must be 1 or 2.");
  TORCH_CHECK(gate.scalar_type() == at::kFloat, "gate must be float32.");
  TORCH_CHECK(is_16bit(x), "x must be float16 or bfloat16.");
  const int64_t B = x.size(0), H = x.size(1), L = x.size(3);
  TORCH_CHECK(L % 16 == 0, "Length L must be multiple of 16");
  check_layout("gate", gate, {B, H, L});
  check_layout("x", x, {B, H, 16, L});
}

// y <- btp(exp(gate), x), the exponential taken in fp32 inside the kernel (no reference counterpart).
void forward_log(const at::Tensor& gate, const at::Tensor& x, at::Tensor y, int64_t k) {
  check_log_common(gate, x, k);
  const int64_t B = x.size(0), H = x.size(1), L = x.size(3);
  TORCH_CHECK(y.is_cuda(), "All tensors must be CUDA.");
  TORCH_CHECK(y.scalar_type() == at::kFloat || y.scalar_type() == x.scalar_type(), "y must be float32 or match x dtype.");
  check_layout("y", y, {B, H, 16, L});
  check_same_device({&gate, &x, &y});
  const c10::DeviceGuard guard(x.device());
  const int rc = spear_btp_forward_loggate(static_cast<const float*>(gate.data_ptr()), x.data_ptr(), y.data_ptr(), nullptr,
                                           (int)B, (int)H, (int)L, (int)k, tag_of(x.scalar_type()),
                                           tag_of(y.scalar_type()), 0u, stream_of(x));
  if (rc != 0) raise_native(rc);
}

// dx, dgate <- vjp of btp(exp(gate), x); a float32 dx selects the fp32 check mode.
void backward_log(const at::Tensor& gate, const at::Tensor& x, const at::Tensor& dy, at::Tensor dx, at::Tensor dgate,
                  int64_t k) {
  check_log_common(gate, x, k);
  const int64_t B = x.size(0), H = x.size(1), L = x.size(3);
  TORCH_CHECK(dy.is_cuda() && dx.is_cuda() && dgate.is_cuda(), "All tensors must be CUDA.");
  TORCH_CHECK(dx.scalar_type() == x.scalar_type() || dx.scalar_type() == at::kFloat, "dx must be float32 or match x dtype.");
  TORCH_CHECK(dgate.scalar_type() == at::kFloat, "dgate must be float32.");
  TORCH_CHECK(dy.scalar_type() == at::kFloat || dy.scalar_type() == x.scalar_type(), "dy must be float32 or match x dtype.");
  check_layout("dy", dy, {B, H, 16, L});
  check_layout("dx", dx, {B, H, 16, L});
  check_layout("dgate", dgate, {B, H, L});
  check_same_device({&gate, &x, &dy, &dx, &dgate});
  const c10::DeviceGuard guard(x.device());
  const unsigned flags = dx.scalar_type() == at::kFloat ? SPEAR_BTP_DX_F32 : 0u;
  const int rc = spear_btp_backward_loggate(static_cast<const float*>(gate.data_ptr()), x.data_ptr(), dy.data_ptr(),
                                            dx.data_ptr(), static_cast<float*>(dgate.data_ptr()), (int)B, (int)H, (int)L,
                                            (int)k, tag_of(x.scalar_type()), tag_of(dy.scalar_type()), flags, stream_of(x));
  if (rc != 0) raise_native(rc);
}

// The autograd node of btp(), compiled: forward allocates y (and the checkpoint, a zero-element placeholder
// unless the store is on), backward allocates dx and dA, both call the functions above. It does what
// _BTPFunction of the reference does (spear/ops/btp/interface.py:126-161) without the Python frames of
// torch.autograd.Function and of the custom-op dispatch, which at small batches cost several times the
// kernels' time. The Python side uses it for plain eager tensors only; under torch.compile and dispatch modes
// the Python node over the traceable custom ops runs instead.
struct BtpNode : public torch::autograd::Function<BtpNode> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& coeff, const at::Tensor& x, int64_t k,
                            int64_t wpb, bool y_f32, int64_t forward_flags, int64_t backward_flags) {
    TORCH_CHECK(x.dim() == 4, "x must be [B, H, 16, L].");
    at::Tensor y = at::empty(x.sizes(), x.options().dtype(y_f32 ? at::kFloat : x.scalar_type()));
    at::Tensor checkpoint =
        (forward_flags & SPEAR_BTP_WRITE_CHECKPOINT)
            ? at::empty({x.size(0), x.size(1), x.size(3) / 16, 16}, x.options().dtype(at::kFloat))
            : at::empty({0}, x.options().dtype(at::kFloat));
    ::forward(coeff, x, y, checkpoint, k, wpb, forward_flags);
    ctx->save_for_backward({coeff, x, checkpoint});
    ctx->saved_data["k"] = k;
    ctx->saved_data["wpb"] = wpb;
    ctx->saved_data["flags"] = backward_flags;
    return y;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grad_outputs) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &coeff = saved[0], &x = saved[1], &checkpoint = saved[2];
    const at::Tensor dy = grad_outputs[0].contiguous();
    at::Tensor dx = at::empty(x.sizes(), x.options());
    // The engine hands the gradient on in coeff's dtype; the kernel can round it there itself (the matrix-core path
    // stores fp32 and leaves the rounding to the engine).
    int64_t flags = ctx->saved_data["flags"].toInt();
    if (!(flags & SPEAR_BTP_PATH_MFMA)) flags |= SPEAR_BTP_DA_16;
    at::Tensor dA = at::empty(coeff.sizes(), (flags & SPEAR_BTP_DA_16) ? coeff.options() : coeff.options().dtype(at::kFloat));
    ::backward(coeff, x, dy, checkpoint, dx, dA, ctx->saved_data["k"].toInt(), ctx->saved_data["wpb"].toInt(), flags);
    return {dA, dx, at::Tensor(), at::Tensor(), at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

at::Tensor btp_autograd(const at::Tensor& coeff, const at::Tensor& x, int64_t k, int64_t wpb, bool y_f32,
                        int64_t forward_flags, int64_t backward_flags) {
  return BtpNode::apply(coeff, x, k, wpb, y_f32, forward_flags, backward_flags);
}

struct MixShape {
  int64_t B, L, F, Fkv;
};

MixShape check_mix_shapes(const at::Tensor& a_logit, const at::Tensor& b_logit, const at::Tensor& c, const at::Tensor& v,
                          int64_t heads, int64_t kv_heads, bool qkv_gate) {
  TORCH_CHECK(a_logit.is_cuda() && b_logit.is_cuda() && c.is_cuda() && v.is_cuda(), "All tensors must be CUDA.");
  TORCH_CHECK(v.dim() == 3 && v.size(2) == heads * 16, "v must be [B, L, heads * 16].");
  TORCH_CHECK(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "heads must be divisible by kv_heads.");
  TORCH_CHECK(is_16bit(v), "tensors must be float16 or bfloat16.");
  TORCH_CHECK(b_logit.scalar_type() == v.scalar_type() && c.scalar_type() == v.scalar_type(), "all tensors must share one dtype.");
  if (qkv_gate) {
    TORCH_CHECK(a_logit.scalar_type() == at::kFloat, "the log-decay gate must be float32.");
  } else {
    TORCH_CHECK(a_logit.scalar_type() == v.scalar_type(), "all tensors must share one dtype.");
  }
  const MixShape s{v.size(0), v.size(1), v.size(2), kv_heads * 16};
  check_layout("a_logit", a_logit, {s.B, s.L, heads});
  check_layout("b_logit", b_logit, {s.B, s.L, s.Fkv});
  check_layout("c", c, {s.B, s.L, s.Fkv});
  check_layout("v", v, {s.B, s.L, s.F});
  return s;
}

MixShape check_mix_inputs(const at::Tensor& a_logit, const at::Tensor& b_logit, const at::Tensor& c, const at::Tensor& v,
                          int64_t heads, int64_t kv_heads, bool qkv_gate) {
  const MixShape s = check_mix_shapes(a_logit, b_logit, c, v, heads, kv_heads, qkv_gate);
  TORCH_CHECK(s.L % 16 == 0, "Length L must be multiple of 16");
  return s;
}

// out <- btp(sigmoid(a_logit), sigmoid(b_logit) * v) * c + v on [B, L, features] tensors, or with
// qkv_gate out <- c * btp(exp(a_logit), b_logit * v) + v. A float32 `out` selects the fp32 check mode.
void mix_forward(const at::Tensor& a_logit, const at::Tensor& b_logit, const at::Tensor& c, const at::Tensor& v,
                 at::Tensor out, int64_t heads, int64_t kv_heads, bool qkv_gate, bool round_products = false) {
  const MixShape s = check_mix_inputs(a_logit, b_logit, c, v, heads, kv_heads, qkv_gate);
  TORCH_CHECK(out.is_cuda(), "All tensors must be CUDA.");
  TORCH_CHECK(out.scalar_type() == v.scalar_type() || out.scalar_type() == at::kFloat,
              "out must be float32 (fp32 check mode) or match v dtype.");
  check_layout("out", out, {s.B, s.L, s.F});
  check_same_device({&a_logit, &b_logit, &c, &v, &out});
  const c10::DeviceGuard guard(v.device());
  const unsigned flags = (qkv_gate ? SPEAR_MIX_QKV_GATE : 0u) | (out.scalar_type() == at::kFloat ? SPEAR_MIX_F32_RESULTS : 0u) |
                         (round_products ? SPEAR_MIX_ROUND : 0u);
  const int rc = spear_phalanx_mix_forward(a_logit.data_ptr(), b_logit.data_ptr(), c.data_ptr(), v.data_ptr(), out.data_ptr(),
                                           (int)s.B, (int)s.L, (int)heads, (int)kv_heads, tag_of(v.scalar_type()), flags,
                                           stream_of(v));
  if (rc != 0) raise_native(rc);
}

// Elements per time step of a [B, L, width] tensor that is dense or a column block of a wider buffer.
int64_t row_stride(const char* name, const at::Tensor& t, int64_t B, int64_t L, int64_t width) {
  TORCH_CHECK(t.dim() == 3 && t.size(0) == B && t.size(1) == L && t.size(2) == width, name, " must have shape [", B, ", ",
              L, ", ", width, "], got ", t.sizes(), ".");
  const int64_t ld = L > 1 ? t.stride(1) : (B > 1 ? t.stride(0) : width);
  TORCH_CHECK(t.stride(2) == 1 && (L <= 1 || t.stride(1) == ld) && (B <= 1 || t.stride(0) == L * ld), name,
              " must be dense or a column block of a dense [B, L, ld] buffer.");
  return ld;
}

// Gradients of mix_forward, written in place. Float32 db_logit / dc / dv (and da_logit) select the fp32
// check mode. `sums`: none, or three fp32 [rows, width] tensors receiving the column sums of every (batch row,
// tile of 64 time steps).
void mix_backward(const at::Tensor& a_logit, const at::Tensor& b_logit, const at::Tensor& c, const at::Tensor& v,
                  const at::Tensor& dout, at::Tensor da_logit, at::Tensor db_logit, at::Tensor dc, at::Tensor dv,
                  int64_t heads, int64_t kv_heads, const std::vector<at::Tensor>& sums, bool qkv_gate, bool round_products = false) {
  const MixShape s = check_mix_inputs(a_logit, b_logit, c, v, heads, kv_heads, qkv_gate);
  TORCH_CHECK(dout.is_cuda() && da_logit.is_cuda() && db_logit.is_cuda() && dc.is_cuda() && dv.is_cuda(), "All tensors must be CUDA.");
  TORCH_CHECK(dout.scalar_type() == v.scalar_type(), "all tensors must share one dtype.");
  check_layout("dout", dout, {s.B, s.L, s.F});
  const bool f32 = dv.scalar_type() == at::kFloat;
  TORCH_CHECK(db_logit.scalar_type() == dv.scalar_type() && dc.scalar_type() == dv.scalar_type() &&
                  (f32 || dv.scalar_type() == v.scalar_type()),
              "db_logit, dc and dv must all be float32 (fp32 check mode) or all match v dtype.");
  if (qkv_gate || f32) {
    TORCH_CHECK(da_logit.scalar_type() == at::kFloat, "the gradient of the gate must be float32.");
  } else {
    TORCH_CHECK(da_logit.scalar_type() == v.scalar_type(), "all tensors must share one dtype.");
  }
  TORCH_CHECK(sums.empty() || sums.size() == 3, "sums must be three tensors or none.");
  TORCH_CHECK(sums.empty() || !qkv_gate, "column sums belong to the layer form, not to qkv_gate.");
  TORCH_CHECK(sums.empty() || !f32, "column sums are not available in the fp32 check mode.");
  const int64_t ld_da = row_stride("da_logit", da_logit, s.B, s.L, heads), ld_db = row_stride("db_logit", db_logit, s.B, s.L, s.Fkv),
                ld_dc = row_stride("dc", dc, s.B, s.L, s.Fkv), ld_dv = row_stride("dv", dv, s.B, s.L, s.F);
  check_same_device({&a_logit, &b_logit, &c, &v, &dout, &da_logit, &db_logit, &dc, &dv});
  int64_t rows = 0;
  float* sp[3] = {nullptr, nullptr, nullptr};
  if (!sums.empty()) {
    rows = spear_phalanx_mix_backward_sum_rows((int)s.B, (int)s.L, (int)heads);
    const int64_t widths[3] = {heads, s.Fkv, s.Fkv};
    const char* names[3] = {"sum_da", "sum_db", "sum_dc"};
    for (int i = 0; i < 3; ++i) {
      TORCH_CHECK(sums[i].is_cuda() && sums[i].device() == v.device() && sums[i].scalar_type() == at::kFloat, names[i],
                  " must be float32 on v's device.");
      check_layout(names[i], sums[i], {rows, widths[i]});
      sp[i] = rows > 0 ? static_cast<float*>(sums[i].data_ptr()) : nullptr;
    }
  }
  const c10::DeviceGuard guard(v.device());
  const unsigned flags = (qkv_gate ? SPEAR_MIX_QKV_GATE : 0u) | (f32 ? SPEAR_MIX_F32_RESULTS : 0u) | (round_products ? SPEAR_MIX_ROUND : 0u);
  const int rc = spear_phalanx_mix_backward_ex(
      a_logit.data_ptr(), b_logit.data_ptr(), c.data_ptr(), v.data_ptr(), dout.data_ptr(), da_logit.data_ptr(),
      db_logit.data_ptr(), dc.data_ptr(), dv.data_ptr(), (int)ld_da, (int)ld_db, (int)ld_dc, (int)ld_dv, sp[0], sp[1], sp[2],
      rows, (int)s.B, (int)s.L, (int)heads, (int)kv_heads, tag_of(v.scalar_type()), flags, stream_of(v));
  if (rc != 0) raise_native(rc);
}

// The autograd node of btp_log(), compiled like BtpNode: forward allocates y, backward dx and dgate.
struct BtpLogNode : public torch::autograd::Function<BtpLogNode> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& gate, const at::Tensor& x, int64_t k,
                            bool y_f32) {
    TORCH_CHECK(x.dim() == 4, "x must be [B, H, 16, L].");
    at::Tensor y = at::empty(x.sizes(), x.options().dtype(y_f32 ? at::kFloat : x.scalar_type()));
    forward_log(gate, x, y, k);
    ctx->save_for_backward({gate, x});
    ctx->saved_data["k"] = k;
    return y;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grad_outputs) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &gate = saved[0], &x = saved[1];
    at::Tensor dx = at::empty(x.sizes(), x.options());
    at::Tensor dgate = at::empty(gate.sizes(), gate.options());
    backward_log(gate, x, grad_outputs[0].contiguous(), dx, dgate, ctx->saved_data["k"].toInt());
    return {dgate, dx, at::Tensor(), at::Tensor()};
  }
};

at::Tensor btp_log_autograd(const at::Tensor& gate, const at::Tensor& x, int64_t k, bool y_f32) {
  return BtpLogNode::apply(gate, x, k, y_f32);
}

// The autograd node of phalanx_mix() and, with qkv_gate, of btp_qkv() (operands then in the kernel's order: gate,
// k, q, v), compiled: forward allocates out, backward the four gradients (the first one in a_logit's dtype, which
// for the q/k/v/gate form is the fp32 of the gate). What spear_amd/ops/btp/fused.py does in torch.autograd.Function
// classes over the traceable custom ops, without their Python frames; used for plain eager tensors only.
struct MixNode : public torch::autograd::Function<MixNode> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& a_logit, const at::Tensor& b_logit,
                            const at::Tensor& c, const at::Tensor& v, int64_t heads, int64_t kv_heads, bool qkv_gate) {
    at::Tensor out = at::empty(v.sizes(), v.options());
    mix_forward(a_logit, b_logit, c, v, out, heads, kv_heads, qkv_gate);
    ctx->save_for_backward({a_logit, b_logit, c, v});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["kv_heads"] = kv_heads;
    ctx->saved_data["qkv_gate"] = qkv_gate;
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grad_outputs) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &a_logit = saved[0], &b_logit = saved[1], &c = saved[2], &v = saved[3];
    at::Tensor da = at::empty(a_logit.sizes(), a_logit.options()), db = at::empty(b_logit.sizes(), b_logit.options()),
               dc = at::empty(c.sizes(), c.options()), dv = at::empty(v.sizes(), v.options());
    mix_backward(a_logit, b_logit, c, v, grad_outputs[0].contiguous(), da, db, dc, dv, ctx->saved_data["heads"].toInt(),
                 ctx->saved_data["kv_heads"].toInt(), {}, ctx->saved_data["qkv_gate"].toBool());
    return {da, db, dc, dv, at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

at::Tensor mix_autograd(const at::Tensor& a_logit, const at::Tensor& b_logit, const at::Tensor& c, const at::Tensor& v,
                        int64_t heads, int64_t kv_heads, bool qkv_gate) {
  return MixNode::apply(a_logit, b_logit, c, v, heads, kv_heads, qkv_gate);
}

// A prompt through the mixing stage: out and the streaming state after it (h, r, c_prev, pos), all allocated here. Any L >= 1.
std::vector<at::Tensor> mix_prefill(const at::Tensor& a_logit, const at::Tensor& b_logit, const at::Tensor& c, const at::Tensor& v,
                                    int64_t heads, int64_t kv_heads) {
  const MixShape s = check_mix_shapes(a_logit, b_logit, c, v, heads, kv_heads, false);
  check_same_device({&a_logit, &b_logit, &c, &v});
  const auto f32 = v.options().dtype(at::kFloat);
  at::Tensor out = at::empty_like(v), h = at::empty({s.B, heads, 16}, f32), r = at::empty({s.B, heads}, f32),
             c_prev = at::empty({s.B, heads, 16}, f32), pos = at::empty({s.B}, v.options().dtype(at::kInt));
  const c10::DeviceGuard guard(v.device());
  const int rc = spear_layer_prefill(a_logit.data_ptr(), b_logit.data_ptr(), c.data_ptr(), v.data_ptr(), out.data_ptr(),
                                     h.data_ptr<float>(), r.data_ptr<float>(), c_prev.data_ptr<float>(), pos.data_ptr<int>(),
                                     (int)s.B, (int)s.L, (int)heads, (int)kv_heads, tag_of(v.scalar_type()), stream_of(v));
  if (rc != 0) raise_native(rc);
  return {out, h, r, c_prev, pos};
}

// out[i] <- column sums of the dense fp32 matrix in[i], rounded to out[i]'s 16-bit type: one launch for all.
void layer_sums(const std::vector<at::Tensor>& in, const std::vector<at::Tensor>& out) {
  TORCH_CHECK(in.size() == out.size() && !in.empty() && in.size() <= 5, "1 to 5 matrices with a result each.");
  const float* src[5];
  void* dst[5];
  long long rows[5], cols[5];
  for (size_t i = 0; i < in.size(); ++i) {
    TORCH_CHECK(in[i].is_cuda() && out[i].is_cuda() && in[i].dim() == 2 && in[i].scalar_type() == at::kFloat, "matrices must be float32 CUDA tensors.");
    TORCH_CHECK(is_16bit(out[i]) && out[i].scalar_type() == out[0].scalar_type(), "results must be float16 or bfloat16, all of one type.");
    TORCH_CHECK(in[i].is_contiguous() && out[i].is_contiguous() && out[i].numel() == in[i].size(1), "matrices and results must be dense, one result per column.");
    check_same_device({&in[0], &in[i], &out[i]});
    src[i] = static_cast<const float*>(in[i].data_ptr());
    dst[i] = out[i].data_ptr();
    rows[i] = in[i].size(0);
    cols[i] = in[i].size(1);
  }
  const c10::DeviceGuard guard(in[0].device());
  const int rc = spear_layer_sums((int)in.size(), src, dst, rows, cols, tag_of(out[0].scalar_type()), stream_of(in[0]));
  if (rc != 0) raise_native(rc);
}

// x [..., K] through up to four linear layers in one launch (bf16; biases may be undefined): [..., N_i] each, allocated in that shape (a
// view of a matrix would leave an autograd node as a view, on which callers could not work in place). x dense, or [M, K] with dense rows.
std::vector<at::Tensor> linears(const at::Tensor& x, const std::vector<at::Tensor>& weights, const std::vector<at::Tensor>& biases,
                                int* pos = nullptr, int64_t block_len = 0) {
  TORCH_CHECK(x.is_cuda() && x.dim() >= 2 && x.scalar_type() == at::kBFloat16, "x must be a bfloat16 CUDA tensor of two dimensions or more.");
  const bool rows = x.dim() == 2;
  TORCH_CHECK(rows ? x.stride(1) == 1 : x.is_contiguous(), "x must have dense rows, and be dense where it has more than two dimensions.");
  TORCH_CHECK(!weights.empty() && weights.size() <= 4 && biases.size() == weights.size(), "1 to 4 layers.");
  const int64_t K = x.size(-1), M = K > 0 ? x.numel() / K : 0;
  const void *w[4], *b[4];
  void* o[4];
  int N[4];
  std::vector<at::Tensor> out;
  std::vector<int64_t> sizes = x.sizes().vec();
  for (size_t i = 0; i < weights.size(); ++i) {
    const int64_t n = weights[i].size(0);
    check_layout("weight", weights[i], {n, K});
    TORCH_CHECK(weights[i].scalar_type() == at::kBFloat16, "weights must be bfloat16.");
    if (biases[i].defined()) {
      check_layout("bias", biases[i], {n});
      TORCH_CHECK(biases[i].scalar_type() == at::kBFloat16, "biases must be bfloat16.");
    }
    check_same_device({&x, &weights[i], &biases[i]});
    sizes.back() = n;
    out.push_back(at::empty(sizes, x.options()));
    w[i] = weights[i].data_ptr();
    b[i] = biases[i].defined() ? biases[i].data_ptr() : nullptr;
    o[i] = out[i].data_ptr();
    N[i] = (int)n;
  }
  const c10::DeviceGuard guard(x.device());
  const int rc = spear_layer_linear((int)weights.size(), x.data_ptr(), rows && M > 1 ? x.stride(0) : K, (int)M, (int)K, w, b, o, N, pos, (int)block_len,
                                    stream_of(x));
  if (rc != 0) raise_native(rc);
  return out;
}

// Whether projections of M rows are faster through spear_layer_linear than as the library's products. Measured in HIP graphs, us, dim = K,
// spear_layer_linear / the library. The four input projections: K=128 131072 rows 49 / 67, K=512 1024 rows 8 / 22, 131072 rows 229 / 284,
// K=768 65536 rows 230 / 239, K=1024 8192 rows 54 / 72, 131072 rows 729 / 717 (with kv heads shared by four 401 / 405), K=1536 16384 rows
// 203 / 238, 65536 rows 772 / 742, K=2048 4096 rows 95 / 114, 8192 rows 193 / 174: all below K = 1024, and few tiles from there on.
// One: K=512 65536 rows 40 / 43, 16384 rows 13.7 / 15.5, K=1024 16 rows 4.3 / 4.2, 1024 rows 10.6 / 7.7, 4096 rows 13.5 / 13.5, 16384 rows 34 / 30,
// K=2048 16 rows 6.0 / 5.3, 1024 rows 19 / 15, K=4096 16 rows 10 / 11, 512 rows 33 / 24. On the GPU it is mostly up to 4 us slower up to 9 G
// multiply-adds, and saves the 15 us that a library product costs the host, which is what bounds calls of that size. The tiles start at K = 72; up to 64 the few-row kernel is left, which reads its operands too often for
// many rows (a layer's forward at 1048576 rows, it / the library: K=32 541 / 384, K=64 838 / 470; 8192 rows within 5 %).
bool own_products(int64_t M, const std::vector<at::Tensor>& weights, int64_t K) {
  if (M <= 0 || K <= 0 || K % 8 != 0) return false;
  if (K <= 64) {
    int64_t columns = 0;
    for (const at::Tensor& w : weights) columns += w.size(0);
    return M * columns * K <= (weights.size() > 1 ? 1600000000 : 300000000);
  }
  if (weights.size() == 1) return K <= 512 || M * weights[0].size(0) * K <= 9000000000;
  int64_t tiles = 0;
  for (const at::Tensor& w : weights) tiles += (w.size(0) + 255) / 256;
  tiles *= (M + 255) / 256;
  return K < 1024 || tiles <= 600;
}

// The four input projections (a, b, c, v) of x [..., K], or one projection without bias, by either. x dense.
std::vector<at::Tensor> project(const at::Tensor& x, const std::vector<at::Tensor>& weights, const std::vector<at::Tensor>& biases) {
  const int64_t K = x.size(-1), M = K > 0 ? x.numel() / K : 0;
  if (own_products(M, weights, K) && (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15u) == 0) return linears(x, weights, biases);
  std::vector<at::Tensor> out;
  for (size_t i = 0; i < weights.size(); ++i) out.push_back(biases[i].defined() ? at::linear(x, weights[i], biases[i]) : at::linear(x, weights[i]));
  return out;
}

// dy [M, N], x [M, K] -> dy^T x [N, K] in dy's type, fp32 sums. With s > 1 the token axis is cut into s slices multiplied as one
// batched product with fp32 parts, which the caller adds with layer_sums (`parts`, `sums`).
at::Tensor weight_grad(const at::Tensor& dy, const at::Tensor& x, int64_t s, std::vector<at::Tensor>& parts, std::vector<at::Tensor>& sums) {
  const int64_t M = dy.size(0), N = dy.size(1), K = x.size(1);
  if (s <= 1) return at::mm(dy.t(), x);
  at::Tensor out = at::empty({N, K}, dy.options());
  parts.push_back(at::bmm(dy.view({s, M / s, N}).transpose(1, 2), x.view({s, M / s, K}), at::kFloat).view({s, N * K}));
  sums.push_back(out);
  return out;
}

// Weight gradients of one backward pass through spear_layer_wgrad: products dy^T x in one launch, the sums of those cut into splits and the bias
// gradients' in another.
struct WeightGrads {
  std::vector<at::Tensor> dy, x, dw;  // dy [M, N or more], x [M, K], dw [N, K]
  std::vector<int> slices;            // of the tokens, that the library's product would have: at least as many splits

  void add(const at::Tensor& grad, const at::Tensor& operand, int64_t columns, int64_t least) {
    slices.push_back((int)least);
    dy.push_back(grad);
    x.push_back(operand);
    dw.push_back(at::empty({columns, operand.size(1)}, operand.options()));
  }

  void run(const std::vector<at::Tensor>& sums_of, const std::vector<at::Tensor>& sums) {
    const int n = (int)dy.size();
    const void *g[2], *o[2];
    void *whole[2], *w[2];
    int ld[2], N[2], K[2], splits[2], rows_of[2], cols_of[2], splits_of[2], parted = 0;  // w and *_of: the products with parts
    const int64_t M = x[0].size(0);
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) {
      g[i] = dy[i].data_ptr();
      o[i] = x[i].data_ptr();
      ld[i] = (int)dy[i].size(1);
      N[i] = (int)dw[i].size(0);
      K[i] = (int)dw[i].size(1);
      splits[i] = spear_layer_wgrad_splits_from(M, N[i], K[i], slices[i]);
      whole[i] = splits[i] == 1 && K[i] < 1 << 21 ? dw[i].data_ptr() : nullptr;
      if (whole[i] != nullptr) continue;
      blocks += (int64_t)((N[i] + 255) / 256) * ((K[i] + 255) / 256) * splits[i];
      rows_of[parted] = N[i];
      cols_of[parted] = K[i];
      splits_of[parted] = splits[i];
      w[parted++] = dw[i].data_ptr();
    }
    at::Tensor parts;
    if (blocks > 0) parts = at::empty({blocks * 65536}, x[0].options().dtype(at::kFloat));
    float* const to = blocks > 0 ? static_cast<float*>(parts.data_ptr()) : nullptr;
    int rc = spear_layer_wgrad_to(n, g, ld, ld, N, o, K, splits, M, to, whole, stream_of(x[0]));
    if (rc != 0) raise_native(rc);
    if (parted == 0) {
      if (!sums.empty()) layer_sums(sums_of, sums);
      return;
    }
    const float* in[3];
    void* out[3];
    long long rows[3], cols[3];
    for (size_t i = 0; i < sums.size(); ++i) {
      in[i] = static_cast<const float*>(sums_of[i].data_ptr());
      out[i] = sums[i].data_ptr();
      rows[i] = sums_of[i].size(0);
      cols[i] = sums_of[i].size(1);
    }
    rc = spear_layer_wgrad_sums(parted, to, rows_of, cols_of, splits_of, w, (int)sums.size(), in, out, rows, cols, SPEAR_BTP_BF16, stream_of(x[0]));
    if (rc != 0) raise_native(rc);
  }
};

// Whether the weight gradients of a layer's backward are faster through spear_layer_wgrad than as the library's (sliced) products: up to
// 32768 tokens, and above from 12 G multiply-adds on. Times of single products at layer_wgrad.hip. A whole step, us (and on the GPU alone),
// with them here / the library's: 1024 tokens, width 512 124 (86) / 169 (86), 4096 tokens 257 (116) / 291 (134), 1024 tokens, width 1024 259
// (129) / 298 (130), 131072 tokens, width 128 287 / 280. Up to 1024 tokens they are the slower ones on the GPU (both of a layer at width 512 16 / 9
// us, 1024 16 / 11, 2048 27 / 19 at 64 tokens, 24 / 23, 33 / 28, 65 / 52 at 1024) and save the host 30 us, which bounds such a step.
bool own_weight_grads(int64_t M, int64_t multiply_adds_per_token) { return M <= 32768 || M * multiply_adds_per_token >= 12000000000; }

// Few tokens of a very wide layer, whose step the GPU bounds: there the library's products are the faster ones for all gradients; it takes the
// weights as they lie, and transposing them reads and writes each once more. A step, us, with the library's / here:
// 68 M weights (width 4096, kv heads its own) 64 tokens 299 / 309, 256 304 / 394, 512 400 / 489, 1024 550 / 595, 2048 880 / 966, 4096 1489 / 1478;
// 43 M (width 4096, shared by four) 128 tokens 241 / 216, 256 238 / 252, 512 252 / 288, 2048 553 / 598, 4096 974 / 945; 38 M (width 3072) 128 tokens 307 / 213, 512
// 305 / 314, 1024 397 / 373, 2048 577 / 609; 17 M (width 2048) 512 tokens 227 / 181, 1024 229 / 227; 270 M (width 8192) 64 tokens 720 / 1037, 2048 2860 / 2972. In a
// graph the library's would be the faster ones in narrower layers too (17 M weights, 512 tokens 152 / 181; 38 M, 256 216 / 250).
bool few_tokens_of_many_weights(int64_t M, int64_t weights) { return M <= 2048 && (weights >= 60000000 || (weights >= 40000000 && M >= 256)); }

// A whole layer call on plain bf16 tensors: the four input projections, the mixing stage and the output projection, with one
// autograd node. Backward is what spear_amd/nn/phalanx/projections.py does with _ProjectAndMix and _Linear (one product each for the
// input and weight gradients of the four projections, against the packed gradient buffer), without Python frames and with
// layer_transpose and layer_sums around the products: 9 launches for forward and backward of a small layer where separate modules had 29.
// The mixing kernels are the same.
struct LayerNode : public torch::autograd::Function<LayerNode> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& x, const at::Tensor& w_a, const at::Tensor& b_a,
                            const at::Tensor& w_b, const at::Tensor& b_b, const at::Tensor& w_c, const at::Tensor& b_c,
                            const at::Tensor& w_v, const at::Tensor& w_out, int64_t heads, int64_t kv_heads, int64_t slices_in,
                            int64_t slices_out, bool round_products) {
    const auto front = project(x, {w_a, w_b, w_c, w_v}, {b_a, b_b, b_c, at::Tensor()});
    const at::Tensor &a = front[0], &b = front[1], &c = front[2], &v = front[3];
    at::Tensor mixed = at::empty(v.sizes(), v.options());
    mix_forward(a, b, c, v, mixed, heads, kv_heads, false, round_products);
    at::Tensor y = project(mixed, {w_out}, {at::Tensor()})[0];
    if (ctx != nullptr) {
      ctx->save_for_backward({x, w_a, w_b, w_c, w_v, w_out, a, b, c, v, mixed});
      ctx->saved_data["biases"] = std::vector<at::Tensor>{b_a, b_b, b_c};  // for their graphs: their values may change before backward
      ctx->saved_data["heads"] = heads;
      ctx->saved_data["kv_heads"] = kv_heads;
      ctx->saved_data["slices_in"] = slices_in;
      ctx->saved_data["slices_out"] = slices_out;
      ctx->saved_data["round_products"] = round_products;
    }
    return y;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grad_outputs) {
    const bool create_graph = at::GradMode::is_enabled();
    const at::NoGradGuard no_grad;
    const auto saved = ctx->get_saved_variables();
    const int64_t heads = ctx->saved_data["heads"].toInt(), kv_heads = ctx->saved_data["kv_heads"].toInt();
    const int64_t B = grad_outputs[0].size(0), L = grad_outputs[0].size(1), K = grad_outputs[0].size(2);  // the layer's input is as wide
    const int64_t F = heads * 16, Fkv = kv_heads * 16, M = B * L;
    const c10::DeviceGuard guard(grad_outputs[0].device());
    // Saved-tensor hooks may hand back other tensors than were saved: the kernels below take these as they lie.
    auto dense = [&](size_t i, at::IntArrayRef sizes) {
      const at::Tensor& t = saved[i];
      TORCH_CHECK(t.scalar_type() == at::kBFloat16 && t.device() == grad_outputs[0].device() && t.sizes() == sizes,
                  "a saved tensor of a Phalanx layer came back with another type, device or shape.");
      const at::Tensor d = t.contiguous();
      return (reinterpret_cast<uintptr_t>(d.data_ptr()) & 15u) == 0 ? d : d.clone();
    };
    const at::Tensor x2 = dense(0, {B, L, K}).view({M, K}), w_a = dense(1, {heads, K}), w_b = dense(2, {Fkv, K}), w_c = dense(3, {Fkv, K}),
                     w_v = dense(4, {F, K}), w_out = dense(5, {K, F}), a = dense(6, {B, L, heads}), b = dense(7, {B, L, Fkv}),
                     c = dense(8, {B, L, Fkv}), v = dense(9, {B, L, F}), mixed2 = dense(10, {B, L, F}).view({M, F});
    const at::Tensor dy = grad_outputs[0].contiguous().view({M, K});
    torch::autograd::variable_list out(14);  // forward's arguments, of which the first nine are tensors
    std::vector<at::Tensor> parts, sums;
    bool front = false, weights = false;
    for (int i = 0; i < 8; ++i) {
      front = front || ctx->needs_input_grad(i);
      weights = weights || ((i == 1 || i == 3 || i == 5 || i == 7) && ctx->needs_input_grad(i));
    }
    const bool library = few_tokens_of_many_weights(M, (2 * Fkv + 2 * F + heads) * K);
    const bool own_weights = !library && own_weight_grads(M, (ctx->needs_input_grad(8) ? K * F : 0) + (weights ? (2 * Fkv + F + heads) * K : 0));
    WeightGrads grads;
    if (ctx->needs_input_grad(8)) {
      if (own_weights && (reinterpret_cast<uintptr_t>(dy.data_ptr()) & 15u) == 0) {
        grads.add(dy, mixed2, K, ctx->saved_data["slices_out"].toInt());
        out[8] = grads.dw[0];
      } else {
        out[8] = weight_grad(dy, mixed2, ctx->saved_data["slices_out"].toInt(), parts, sums);
        if (!parts.empty()) layer_sums(parts, sums);  // while the parts are in the memory-side cache
        parts.clear();
        sums.clear();
      }
    }
    if (front) {
      const int64_t used = 2 * Fkv + F + heads, ld = (used + 63) / 64 * 64;  // [b | c | v | a | padding]
      // Input gradients against the weights transposed, through spear_layer_linear; as the library's products with the weights as they lie
      // only for a gradient off the 16-byte grid, for few tokens of a very wide layer and for many of a narrow one. Measured, us, spear_layer_linear / the library: proj_out's at K=512 131072 rows 75 / 91,
      // 8192 rows 9 / 12, 1024 rows 6.1 / 7.2, K=1024 131072 rows 251 / 268, 1024 rows 11.2 / 9.7, K=2048 65536 rows 453 / 470, 2048 rows 22 /
      // 26; that of the four input projections at K=512 131072 rows 198 / 208, 1024 rows 14 / 11, K=1024 131072 rows 663 / 697, 4096 rows 30 /
      // 35, 1024 rows 27 / 22, K=2048 65536 rows 1213 / 1299, 1024 rows 51 / 49. The transposing launch takes 3 to 6 us, half of
      // which layer_stack took too. Where it is the slower one on the GPU the host's 15 us per library product count for more.
      // Up to K = 64 (see own_products) a step of 131072 tokens takes 324 / 260 us at K=32 and 335 / 285 at K=48, of 8192 tokens 220 / 253.
      const bool own = !library && K % 8 == 0 && (K > 64 || M <= 32768) && (reinterpret_cast<uintptr_t>(dy.data_ptr()) & 15u) == 0;
      const at::Tensor packed = at::empty({B, L, ld}, v.options());
      const at::Tensor stacked = own ? at::empty({K, ld}, v.options()) : at::empty({ld, K}, v.options());
      at::Tensor dmixed;
      if (own) {
        const at::Tensor out_t = at::empty({F, K}, v.options());
        const int rc = spear_layer_transpose(w_a.data_ptr(), w_b.data_ptr(), w_c.data_ptr(), w_v.data_ptr(), w_out.data_ptr(), stacked.data_ptr(),
                                             out_t.data_ptr(), packed.data_ptr(), M, (int)ld, (int)K, (int)heads, (int)Fkv, (int)F, stream_of(v));
        if (rc != 0) raise_native(rc);
        dmixed = linears(dy, {out_t}, {at::Tensor()})[0].view({B, L, F});
      } else {
        const int rc = spear_layer_stack(w_a.data_ptr(), w_b.data_ptr(), w_c.data_ptr(), w_v.data_ptr(), stacked.data_ptr(),
                                         packed.data_ptr(), M, (int)ld, (int)K, (int)heads, (int)Fkv, (int)F, stream_of(v));
        if (rc != 0) raise_native(rc);
        dmixed = at::mm(dy, w_out).view({B, L, F});
      }
      const int64_t rows = spear_phalanx_mix_backward_sum_rows((int)B, (int)L, (int)heads);
      const auto f32 = v.options().dtype(at::kFloat);
      parts = {at::empty({rows, heads}, f32), at::empty({rows, Fkv}, f32), at::empty({rows, Fkv}, f32)};
      mix_backward(a, b, c, v, dmixed, packed.narrow(2, 2 * Fkv + F, heads), packed.narrow(2, 0, Fkv), packed.narrow(2, Fkv, Fkv),
                   packed.narrow(2, 2 * Fkv, F), heads, kv_heads, parts, false, ctx->saved_data["round_products"].toBool());
      sums = {at::empty({heads}, v.options()), at::empty({Fkv}, v.options()), at::empty({Fkv}, v.options())};
      out[2] = sums[0];
      out[4] = sums[1];
      out[6] = sums[2];
      const at::Tensor d2 = packed.view({M, ld});
      if (ctx->needs_input_grad(0)) {
        if (own) {
          out[0] = linears(packed, {stacked}, {at::Tensor()})[0];
        } else {
          out[0] = at::empty({B, L, K}, v.options());  // not a view of the product, for callers that work on it in place
          at::Tensor dx = out[0].view({M, K});
          at::mm_out(dx, d2, stacked);
        }
      }
      if (weights) {
        at::Tensor dw;
        if (own_weights) {
          grads.add(d2, x2, used, ctx->saved_data["slices_in"].toInt());
          dw = grads.dw.back();
        } else {
          dw = weight_grad(d2, x2, ctx->saved_data["slices_in"].toInt(), parts, sums);
        }
        out[3] = dw.narrow(0, 0, Fkv);
        out[5] = dw.narrow(0, Fkv, Fkv);
        out[7] = dw.narrow(0, 2 * Fkv, F);
        out[1] = dw.narrow(0, 2 * Fkv + F, heads);
      }
      if (grads.dy.empty()) layer_sums(parts, sums);
    }
    if (!grads.dy.empty()) grads.run(parts, sums);
    if (!create_graph) return out;
    const at::AutoGradMode grad(true);
    // The mixing kernels have no second derivative: a second differentiation of what their backward has a part in says so.
    const auto twice = twice_differentiable(ctx, saved, grad_outputs[0]);
    torch::autograd::variable_list given;
    std::vector<size_t> at_;
    for (size_t i = 0; i < out.size(); ++i) {
      if (!out[i].defined()) continue;
      if (twice[i].defined()) {
        out[i] = twice[i];
        continue;
      }
      given.push_back(out[i].detach().requires_grad_(true));
      at_.push_back(i);
    }
    const auto error = std::make_shared<torch::autograd::DelayedError>("the gradients of a Phalanx layer cannot be differentiated again", (int64_t)given.size());
    given = error->apply(std::move(given));
    for (size_t i = 0; i < at_.size(); ++i) out[at_[i]] = given[i];
    return out;
  }

  // The gradients that need no backward of the mixing kernels, as functions of the layer's input, its weights and the gradient that
  // arrived: those of proj_out, and of proj_c where the recurrence's result has a tensor of its own (the composition of a default layer).
  static torch::autograd::variable_list twice_differentiable(torch::autograd::AutogradContext* ctx, const torch::autograd::variable_list& saved,
                                                             const at::Tensor& grad_output) {
    torch::autograd::variable_list out(14);
    const bool with_c = ctx->saved_data["round_products"].toBool();
    const bool c_wanted = with_c && (ctx->needs_input_grad(5) || ctx->needs_input_grad(6));
    if (!ctx->needs_input_grad(8) && !c_wanted) return out;
    const at::Tensor &x = saved[0], &w_out = saved[5];
    const int64_t heads = ctx->saved_data["heads"].toInt(), kv_heads = ctx->saved_data["kv_heads"].toInt();
    const int64_t B = x.size(0), L = x.size(1), K = x.size(2), M = B * L, F = heads * 16, Fkv = kv_heads * 16;
    const auto biases = ctx->saved_data["biases"].toTensorVector();
    // the values that forward had, as functions of the input and the weights
    auto projection = [&](const at::Tensor& value, const at::Tensor& w, const at::Tensor& bias) {
      const at::Tensor again = at::linear(x, w, bias);
      return value.detach() + (again - again.detach());
    };
    const at::Tensor a = projection(saved[6], saved[1], biases[0]), b = projection(saved[7], saved[2], biases[1]),
                     c = projection(saved[8], saved[3], biases[2]), v = projection(saved[9], saved[4], at::Tensor()), dy = grad_output.reshape({M, K});
    at::Tensor h, mixed;
    if (with_c) {
      auto expand = [&](const at::Tensor& t) { return t.view({B, L, kv_heads, 1, 16}).expand({B, L, kv_heads, heads / kv_heads, 16}).reshape({B, L, F}); };
      const at::Tensor gated = (expand(at::sigmoid(b)) * v).view({B, L, heads, 16}).permute({0, 2, 3, 1}).contiguous();
      h = BtpNode::apply(at::sigmoid(a).transpose(1, 2).contiguous(), gated, (int64_t)2, (int64_t)32, false, (int64_t)0, (int64_t)0)
              .permute({0, 3, 1, 2}).reshape({B, L, F}).contiguous();
      mixed = h * expand(c) + v;
    } else {
      mixed = MixNode::apply(a, b, c, v, heads, kv_heads, false);
    }
    if (ctx->needs_input_grad(8)) out[8] = at::mm(dy.t(), mixed.view({M, F}));
    if (c_wanted) {
      const at::Tensor dc = (at::mm(dy, w_out).view({B, L, F}) * h).view({M, kv_heads, heads / kv_heads, 16}).sum(2).view({M, Fkv});
      if (ctx->needs_input_grad(5)) out[5] = at::mm(dc.t(), x.reshape({M, K}));
      if (ctx->needs_input_grad(6)) out[6] = dc.sum(0);
    }
    return out;
  }
};

// y = layer(x) for x [B, L, dim]; round_products: gates and products of the mixing stage in 16 bits, as in tensors of their own; slices: into how many slices of tokens the weight gradients' products are cut at least.
at::Tensor layer(const at::Tensor& x, const at::Tensor& w_a, const at::Tensor& b_a, const at::Tensor& w_b, const at::Tensor& b_b,
                 const at::Tensor& w_c, const at::Tensor& b_c, const at::Tensor& w_v, const at::Tensor& w_out, int64_t heads,
                 int64_t kv_heads, int64_t slices_in, int64_t slices_out, bool round_products) {
  TORCH_CHECK(x.dim() == 3 && x.is_contiguous(), "x must be dense [B, L, dim].");
  if (at::GradMode::is_enabled()) {
    for (const at::Tensor* t : {&x, &w_a, &b_a, &w_b, &b_b, &w_c, &b_c, &w_v, &w_out})
      if (t->requires_grad())
        return LayerNode::apply(x, w_a, b_a, w_b, b_b, w_c, b_c, w_v, w_out, heads, kv_heads, slices_in, slices_out, round_products);
  }
  return LayerNode::forward(nullptr, x, w_a, b_a, w_b, b_b, w_c, b_c, w_v, w_out, heads, kv_heads, slices_in, slices_out, round_products);
}

// One token through the layer's input projections and the step of its mixing stage (the caller applies proj_out): x [B, K]
// bf16 with unit column stride, weights and biases of the four projections, the state updated in place.
at::Tensor layer_token(const at::Tensor& x, const at::Tensor& w_a, const at::Tensor& b_a, const at::Tensor& w_b, const at::Tensor& b_b,
                       const at::Tensor& w_c, const at::Tensor& b_c, const at::Tensor& w_v, at::Tensor h, at::Tensor r,
                       at::Tensor c_prev, at::Tensor pos, int64_t block_len, int64_t heads, int64_t kv_heads, bool advance) {
  TORCH_CHECK(x.is_cuda() && h.is_cuda() && r.is_cuda() && c_prev.is_cuda() && pos.is_cuda(), "All tensors must be CUDA.");
  TORCH_CHECK(x.dim() == 2 && x.stride(1) == 1, "x must be [B, dim] with dense rows.");
  TORCH_CHECK(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "heads must be divisible by kv_heads.");
  const int64_t B = x.size(0), K = x.size(1);
  const struct { const char* name; const at::Tensor& t; int64_t rows; } weights[] = {
      {"w_a", w_a, heads}, {"w_b", w_b, kv_heads * 16}, {"w_c", w_c, kv_heads * 16}, {"w_v", w_v, heads * 16}};
  for (const auto& w : weights) check_layout(w.name, w.t, {w.rows, K});
  check_layout("b_a", b_a, {heads});
  check_layout("b_b", b_b, {kv_heads * 16});
  check_layout("b_c", b_c, {kv_heads * 16});
  for (const at::Tensor* t : {&x, &w_a, &b_a, &w_b, &b_b, &w_c, &b_c, &w_v})
    TORCH_CHECK(t->scalar_type() == at::kBFloat16, "x, weights and biases must be bfloat16.");
  TORCH_CHECK(h.scalar_type() == at::kFloat && r.scalar_type() == at::kFloat && c_prev.scalar_type() == at::kFloat, "the state must be float32.");
  TORCH_CHECK(pos.scalar_type() == at::kInt, "pos must be int32.");
  check_layout("h", h, {B, heads, 16});
  check_layout("c_prev", c_prev, {B, heads, 16});
  check_layout("r", r, {B, heads});
  check_layout("pos", pos, {B});
  check_same_device({&x, &w_a, &b_a, &w_b, &b_b, &w_c, &b_c, &w_v, &h, &r, &c_prev, &pos});
  const c10::DeviceGuard guard(x.device());
  at::Tensor out = at::empty({B, heads * 16}, x.options());
  const int rc = spear_layer_token(x.data_ptr(), B > 1 ? x.stride(0) : K, w_a.data_ptr(), b_a.data_ptr(), w_b.data_ptr(), b_b.data_ptr(),
                                   w_c.data_ptr(), b_c.data_ptr(), w_v.data_ptr(), out.data_ptr(), h.data_ptr<float>(),
                                   r.data_ptr<float>(), c_prev.data_ptr<float>(), pos.data_ptr<int>(), (int)block_len, advance ? 1 : 0, (int)B, (int)K,
                                   (int)heads, (int)kv_heads, stream_of(x));
  if (rc != 0) raise_native(rc);
  return out;
}

// A prompt through a whole layer (plain bf16 tensors, x dense [B, L, dim], any L >= 1): [y, h, r, c_prev, pos].
std::vector<at::Tensor> layer_prefill(const at::Tensor& x, const at::Tensor& w_a, const at::Tensor& b_a, const at::Tensor& w_b,
                                      const at::Tensor& b_b, const at::Tensor& w_c, const at::Tensor& b_c, const at::Tensor& w_v,
                                      const at::Tensor& w_out, int64_t heads, int64_t kv_heads) {
  TORCH_CHECK(x.dim() == 3 && x.is_contiguous(), "x must be dense [B, L, dim].");
  const auto front = project(x, {w_a, w_b, w_c, w_v}, {b_a, b_b, b_c, at::Tensor()});
  auto out = mix_prefill(front[0], front[1], front[2], front[3], heads, kv_heads);
  out[0] = project(out[0], {w_out}, {at::Tensor()})[0];
  return out;
}

// One token through a whole layer: layer_token and the output projection.
at::Tensor layer_step(const at::Tensor& x, const at::Tensor& w_a, const at::Tensor& b_a, const at::Tensor& w_b, const at::Tensor& b_b,
                      const at::Tensor& w_c, const at::Tensor& b_c, const at::Tensor& w_v, const at::Tensor& w_out, at::Tensor h,
                      at::Tensor r, at::Tensor c_prev, at::Tensor pos, int64_t block_len, int64_t heads, int64_t kv_heads) {
  // The positions move on with the output projection where that is a kernel of this library: a launch (4.4 us) less, which makes up for what the
  // product takes longer than the library's (see own_products). Not for some tokens of a wide layer: [B, dim] x [dim, dim], us, here / the library's
  // without that launch: dim 3072 B=16 8.2 / 7.4, 64 14.0 / 10.5, 96 19.8 / 13.8; 4096 16 10.2 / 12.1, 32 14.0 / 10.1, 48 17.6 / 11.5, 128 25.8 / 19.6; 6144 16
  // 19.5 / 14.5, 17 21.2 / 15.3, 48 36 / 19.6; 8192 8 23.1 / 22.0, 16 33.6 / 28.0 (in a step). At dim 2048 it is 18.8 / 12.1 for 512 tokens, but the host's time bounds
  // such a step as a call (31 us, 43 with the library's product).
  const auto in = [&](bool advance) { return layer_token(x, w_a, b_a, w_b, b_b, w_c, b_c, w_v, h, r, c_prev, pos, block_len, heads, kv_heads, advance); };
  const int64_t B = x.size(0), K = w_out.size(1);
  const bool wide = K >= 3072 && B >= 16 && B * w_out.size(0) * K >= 500000000;
  if (!wide && own_products(B, {w_out}, K))
    return linears(in(false), {w_out}, {at::Tensor()}, pos.data_ptr<int>(), block_len)[0];
  return at::linear(in(true), w_out);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  namespace py = pybind11;
  m.doc() = "Compiled binding of the MI355X Block Two-Pass library (C ABI of libspear_btp.so)";
  m.def("forward", &forward, py::arg("coeff"), py::arg("x"), py::arg("y"), py::arg("checkpoint"), py::arg("k"), py::arg("wpb"),
        py::arg("flags") = (int64_t)SPEAR_BTP_WRITE_CHECKPOINT, "BTP Forward (HIP, gfx950)");
  m.def("backward", &backward, py::arg("coeff"), py::arg("x"), py::arg("dy"), py::arg("checkpoint"), py::arg("dx"),
        py::arg("dA"), py::arg("k"), py::arg("wpb"), py::arg("flags") = (int64_t)0, "BTP Backward (HIP, gfx950)");
  m.def("btp_autograd", &btp_autograd, py::arg("coeff"), py::arg("x"), py::arg("k"), py::arg("wpb"), py::arg("y_f32"),
        py::arg("forward_flags"), py::arg("backward_flags"),
        "y = btp(coeff, x) with its autograd node (contiguous plain tensors; gradients: dA float32, dx in x's dtype)");
  m.def("forward_log", &forward_log, py::arg("gate"), py::arg("x"), py::arg("y"), py::arg("k"));
  m.def("backward_log", &backward_log, py::arg("gate"), py::arg("x"), py::arg("dy"), py::arg("dx"), py::arg("dgate"), py::arg("k"));
  m.def("mix_forward", &mix_forward, py::arg("a_logit"), py::arg("b_logit"), py::arg("c"), py::arg("v"), py::arg("out"),
        py::arg("heads"), py::arg("kv_heads"), py::arg("qkv_gate") = false, py::arg("round_products") = false);
  m.def("mix_backward", &mix_backward, py::arg("a_logit"), py::arg("b_logit"), py::arg("c"), py::arg("v"), py::arg("dout"),
        py::arg("da_logit"), py::arg("db_logit"), py::arg("dc"), py::arg("dv"), py::arg("heads"), py::arg("kv_heads"),
        py::arg("sums") = std::vector<at::Tensor>(), py::arg("qkv_gate") = false, py::arg("round_products") = false);
  m.def("btp_log_autograd", &btp_log_autograd, py::arg("gate"), py::arg("x"), py::arg("k"), py::arg("y_f32"),
        "y = btp(exp(gate), x) with its autograd node (contiguous plain tensors; gradients: dgate float32, dx in x's dtype)");
  m.def("mix_autograd", &mix_autograd, py::arg("a_logit"), py::arg("b_logit"), py::arg("c"), py::arg("v"), py::arg("heads"),
        py::arg("kv_heads"), py::arg("qkv_gate") = false,
        "out = phalanx_mix(...) (or the q/k/v/gate form) with its autograd node (contiguous plain tensors)");
  m.def("mix_prefill", &mix_prefill, py::arg("a_logit"), py::arg("b_logit"), py::arg("c"), py::arg("v"), py::arg("heads"),
        py::arg("kv_heads"), "[out, h, r, c_prev, pos]: a prompt of any length through the mixing stage, with the state after it");
  m.def("layer", &layer, py::arg("x"), py::arg("w_a"), py::arg("b_a"), py::arg("w_b"), py::arg("b_b"), py::arg("w_c"), py::arg("b_c"),
        py::arg("w_v"), py::arg("w_out"), py::arg("heads"), py::arg("kv_heads"), py::arg("slices_in"), py::arg("slices_out"), py::arg("round_products"),
        "a whole layer call with its autograd node (plain bf16 tensors)");
  m.def("linears", [](const at::Tensor& x, const std::vector<at::Tensor>& w, const std::vector<std::optional<at::Tensor>>& b) {
    std::vector<at::Tensor> biases;
    for (const auto& t : b) biases.push_back(t.value_or(at::Tensor()));
    return linears(x, w, biases);
  }, py::arg("x"), py::arg("weights"), py::arg("biases"), "up to four linear layers on the same rows in one launch (bf16)");
  m.def("layer_prefill", &layer_prefill, "[y, h, r, c_prev, pos]: a prompt through a whole layer (plain bf16 tensors)");
  m.def("layer_step", &layer_step, "one token through a whole layer (plain bf16 tensors), the state updated in place");
  m.def("layer_sums", &layer_sums, py::arg("matrices"), py::arg("results"), "column sums of fp32 matrices, rounded to 16 bits");
  m.def("layer_token", &layer_token, py::arg("x"), py::arg("w_a"), py::arg("b_a"), py::arg("w_b"), py::arg("b_b"), py::arg("w_c"),
        py::arg("b_c"), py::arg("w_v"), py::arg("h"), py::arg("r"), py::arg("c_prev"), py::arg("pos"), py::arg("block_len"),
        py::arg("heads"), py::arg("kv_heads"), py::arg("advance") = true, "one token through the input projections and the step of the mixing stage");
  m.def("abi_version", []() { return spear_btp_abi_version(); });
  m.def("mix_backward_sum_rows", [](int64_t B, int64_t L, int64_t heads) {
    return (int64_t)spear_phalanx_mix_backward_sum_rows((int)B, (int)L, (int)heads);
  }, py::arg("B"), py::arg("L"), py::arg("heads"));
}

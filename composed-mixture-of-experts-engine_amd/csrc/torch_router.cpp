// Native host binding of the router's autograd Function (torch C++ extension `moe_mi355._moe_torch`).
//
// The router step is short on the GPU (C2: ~85 us of kernels for fwd + bwd), so its host work shows: the
// Python Function, eight output allocations through Python, the zeroed-workspace lookup and the ctypes
// conversion of ~25 arguments per call add up to more than the kernels on a slow host.  This file does the
// same work in C++: a torch::autograd::Function whose forward allocates the outputs with ATen, takes the
// current HIP stream from c10 and calls moe_router_fwd, and whose backward (run by the autograd engine
// without returning to Python) calls moe_router_bwd.  It calls the same C ABI entry points
// (include/moe_mi355.h) as the ctypes path and launches the same kernels; argument validation with the
// Python error types stays in moe_mi355/router.py.
//
// The operations that a layer's pass is made of (op_* below) are bound the same way: with few tokens their kernels are
// shorter than the Python that allocates their outputs and converts up to 38 ctypes arguments.  Host work of a pass,
// measured through Python and ctypes -> here: routing 16 bf16 tokens (H 4096, E 8) 24 -> 14 us, a small layer's inference
// 150 -> 122, norm + router with its backward 169 -> 64, dispatch and combine with their backward 169 -> 65, a small
// training step 420 -> 238.
#include <torch/extension.h>

// In torch's ROCm build GPU tensors carry the device type `cuda`; the HIP guard and stream types that accept
// it are the ones "masquerading as CUDA".
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/moe_mi355.h"

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

[[noreturn]] void raise_rc(int rc, const char* what) {
  char buf[512];
  buf[0] = 0;
  moe_last_error(buf, sizeof buf);
  if (rc < 0) throw pybind11::value_error(std::string(what) + ": " + buf + " (code " + std::to_string(rc) + ")");
  throw std::runtime_error(std::string(what) + ": " + buf + " (hip error " + std::to_string(rc) + ")");
}

int code_of(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 ? MOE_BF16 : MOE_F32; }

// The forward's workspace holds a ticket counter that must be zero when a launch starts and that the kernels
// leave at zero: one zero-initialised buffer per (device, stream), reused by every call on that stream.  A call
// may launch several kernels that hand data on through it (the packed gate, the per-block partials), so stream
// order keeps calls apart only if no other thread's launches come between one call's: FwdWorkspace holds the
// buffer's lock until the call's last launch is queued (no call of this file holds the GIL meanwhile, so a
// waiting thread stops no other).
// Under graph capture each capture takes a fresh slice of a per-device arena instead,
// zeroed and synchronised once outside any capture (on the first eager call): the kernels leave the counter at
// zero after every replay, so that slice serves every replay of its graph, and the graph holds no fill node.
// Captures past the arena's end fall back to a zeroed buffer made inside the capture (a captured fill kernel).
struct StreamBuffer {
  std::mutex mu;
  at::Tensor buf;
};
std::mutex g_ws_mu;  // the two maps and the arenas; never held while a StreamBuffer's lock is waited for
std::map<std::pair<int, hipStream_t>, StreamBuffer> g_ws;  // entries stay where they are (a map's nodes)
constexpr int64_t kArenaBytes = 32 << 20;
struct CaptureArena {
  at::Tensor buf;
  int64_t used = 0;
};
std::map<int, CaptureArena> g_arena;

class FwdWorkspace {
 public:
  FwdWorkspace(size_t nbytes, const at::Device& dev, hipStream_t s) {
    const int64_t n = std::max<int64_t>((int64_t)nbytes, 1);
    const auto opts = at::TensorOptions().dtype(at::kByte).device(dev);
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
      (void)hipGetLastError();
      throw std::runtime_error("moe_router_fwd: hipStreamIsCapturing failed");
    }
    StreamBuffer* sb = nullptr;
    {
      std::lock_guard<std::mutex> lk(g_ws_mu);
      CaptureArena& ar = g_arena[(int)dev.index()];
      if (st != hipStreamCaptureStatusNone) {
        const int64_t n256 = (n + 255) / 256 * 256;
        if (ar.buf.defined() && ar.used + n256 <= kArenaBytes) {
          buf_ = ar.buf.narrow(0, ar.used, n);
          ar.used += n256;
        } else {
          buf_ = at::zeros({n}, opts);
        }
        return;
      }
      if (!ar.buf.defined()) {
        ar.buf = at::zeros({kArenaBytes}, opts);
        if (hipStreamSynchronize(s) != hipSuccess) {  // once: later captures may replay on any stream
          (void)hipGetLastError();
          throw std::runtime_error("moe_router_fwd: hipStreamSynchronize failed");
        }
      }
      sb = &g_ws[{(int)dev.index(), s}];
    }
    lock_ = std::unique_lock<std::mutex>(sb->mu);
    if (!sb->buf.defined() || sb->buf.numel() < n) sb->buf = at::zeros({n}, opts);
    buf_ = sb->buf;
  }
  void* data_ptr() const { return buf_.data_ptr(); }

 private:
  at::Tensor buf_;
  std::unique_lock<std::mutex> lock_;
};

struct RouterFn : public torch::autograd::Function<RouterFn> {
  // link_x: x is also returned, as an eighth output, for the layer's expert path to consume.  Its gradient
  // (the expert path's gradient of x) then arrives here as an upstream gradient and is added inside the dx
  // kernel, instead of autograd summing the two contributions to x's gradient in a separate addition.
  static variable_list forward(AutogradContext* ctx, const Variable& x_in, const Variable& gw_in, int64_t k,
                               double aux_coef, double z_coef, const std::optional<Variable>& bias_in, bool link_x) {
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x_in.device());
    const at::Tensor x = x_in.contiguous();
    const at::Tensor gw = gw_in.contiguous();
    const int64_t N = x.size(0), H = x.size(1), E = gw.size(1);
    at::Tensor bias;
    if (bias_in.has_value() && bias_in->defined()) bias = bias_in->detach().to(at::kFloat).contiguous();
    const auto dev = x.device();
    const auto f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
    const auto i64 = at::TensorOptions().dtype(at::kLong).device(dev);
    at::Tensor idx = at::empty({N, k}, i64);
    at::Tensor w = at::empty({N, k}, x.options());
    at::Tensor logits = at::empty({N, E}, f32);
    at::Tensor lse = at::empty({N}, f32);
    at::Tensor cnt = at::empty({E}, i64);
    at::Tensor stats = at::empty({MOE_STATS_HEAD + E}, f32);
    at::Tensor aux = at::empty({}, f32);
    at::Tensor z = at::empty({}, f32);
    if (N == 0) {
      cnt.zero_();
      stats.zero_();
      aux.zero_();
      z.zero_();
    } else {
      const hipStream_t s = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
      const int xdt = code_of(x), wdt = code_of(gw);
      const size_t nbytes = moe_router_fwd_workspace(N, H, E, k, xdt, wdt);
      const FwdWorkspace ws(nbytes, dev, s);
      const int rc = moe_router_fwd(x.data_ptr(), xdt, gw.data_ptr(), wdt,
                                    bias.defined() ? bias.data_ptr<float>() : nullptr, N, H, E, k,
                                    idx.data_ptr<int64_t>(), w.data_ptr(), xdt, logits.data_ptr<float>(),
                                    lse.data_ptr<float>(), cnt.data_ptr<int64_t>(), stats.data_ptr<float>(),
                                    (float)aux_coef, (float)z_coef, aux.data_ptr<float>(), z.data_ptr<float>(),
                                    ws.data_ptr(), nbytes, s);
      if (rc != 0) raise_rc(rc, "moe_router_fwd");
    }
    ctx->save_for_backward({x, gw, logits, idx, cnt});
    ctx->saved_data["aux_coef"] = aux_coef;
    ctx->saved_data["z_coef"] = z_coef;
    ctx->set_materialize_grads(false);
    ctx->mark_non_differentiable({idx, logits, cnt, stats});
    if (link_x) return {idx, w, aux, z, logits, cnt, stats, x_in};
    return {idx, w, aux, z, logits, cnt, stats};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool need_x = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1);
    variable_list out(7);
    if (!(need_x || need_w)) return out;
    const auto saved = ctx->get_saved_variables();
    const at::Tensor& x = saved[0];
    const at::Tensor& gw = saved[1];
    const at::Tensor& logits = saved[2];
    const at::Tensor& idx = saved[3];
    const at::Tensor& cnt = saved[4];
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    at::Tensor g_w = grads[1];
    at::Tensor g_aux = grads[2];
    at::Tensor g_z = grads[3];
    // the linked x output's gradient (the expert path's gradient of x), if any
    at::Tensor dx_add;
    if (need_x && grads.size() > 7 && grads[7].defined()) dx_add = grads[7].to(x.scalar_type()).contiguous();
    const float aux_coef = g_aux.defined() ? (float)ctx->saved_data["aux_coef"].toDouble() : 0.f;
    const float z_coef = g_z.defined() ? (float)ctx->saved_data["z_coef"].toDouble() : 0.f;
    int gdt = MOE_F32;
    if (g_w.defined()) {
      g_w = g_w.contiguous();
      if (g_w.scalar_type() != at::kFloat && g_w.scalar_type() != at::kBFloat16) g_w = g_w.to(at::kFloat);
      gdt = code_of(g_w);
    }
    if (g_aux.defined()) g_aux = g_aux.detach().to(at::kFloat).reshape({1}).contiguous();
    if (g_z.defined()) g_z = g_z.detach().to(at::kFloat).reshape({1}).contiguous();
    const int64_t N = x.size(0), H = x.size(1), E = gw.size(1), K = idx.size(1);
    at::Tensor dx = at::empty({N, H}, x.options());
    at::Tensor dw;
    if (N == 0) {
      dw = at::zeros({H, E}, gw.options());
      dx.zero_();
    } else {
      dw = at::empty({H, E}, gw.options());
      const int xdt = code_of(x), wdt = code_of(gw);
      const size_t nbytes = moe_router_bwd_workspace(N, H, E, K, xdt, wdt);
      const at::Tensor ws = at::empty({std::max<int64_t>((int64_t)nbytes, 1)}, x.options().dtype(at::kByte));
      const hipStream_t s = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index()).stream();
      const int rc = moe_router_bwd_acc(x.data_ptr(), xdt, gw.data_ptr(), wdt, logits.data_ptr<float>(),
                                        idx.data_ptr<int64_t>(), g_w.defined() ? g_w.data_ptr() : nullptr, gdt,
                                        cnt.data_ptr<int64_t>(), g_aux.defined() ? g_aux.data_ptr<float>() : nullptr,
                                        g_z.defined() ? g_z.data_ptr<float>() : nullptr, aux_coef, z_coef, N, H, E, K,
                                        dx_add.defined() ? dx_add.data_ptr() : nullptr, dx.data_ptr(), dw.data_ptr(),
                                        ws.data_ptr(), nbytes, s);
      if (rc != 0) raise_rc(rc, "moe_router_bwd");
    }
    if (need_x) out[0] = dx;
    if (need_w) out[1] = dw;
    return out;
  }
};

variable_list router_core(const at::Tensor& x, const at::Tensor& gate_w, int64_t k, double aux_coef,
                          double z_coef, const std::optional<at::Tensor>& bias, bool link_x) {
  return RouterFn::apply(x, gate_w, k, aux_coef, z_coef, bias, link_x);
}

// ---- the operations of moe_mi355/ops.py: outputs from ATen, one C ABI call, no autograd.  ops.py has checked device,
// types and shapes; tensors arrive as its callers passed them and are made contiguous here where it made them so. ----

using OptTensor = std::optional<at::Tensor>;

hipStream_t stream_of(const at::Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}
const void* ptr(const OptTensor& t) { return t.has_value() && t->defined() ? t->data_ptr() : nullptr; }
at::Tensor scratch(size_t n, const at::Tensor& like) {
  return at::empty({std::max<int64_t>((int64_t)n, 1)}, like.options().dtype(at::kByte));
}
void check_rc(int rc, const char* what) {
  if (rc != 0) raise_rc(rc, what);
}

std::vector<at::Tensor> op_router_forward(const at::Tensor& x_in, const at::Tensor& gw_in, int64_t k, const OptTensor& bias,
                                          bool w_bf16, double aux_coef, double z_coef) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x_in.device());
  const at::Tensor x = x_in.contiguous(), gw = gw_in.contiguous();
  const int64_t N = x.size(0), H = x.size(1), E = gw.size(1);
  const auto f32 = x.options().dtype(at::kFloat);
  const auto i64 = x.options().dtype(at::kLong);
  at::Tensor idx = at::empty({N, k}, i64), w = at::empty({N, k}, x.options().dtype(w_bf16 ? at::kBFloat16 : at::kFloat));
  at::Tensor logits = at::empty({N, E}, f32), lse = at::empty({N}, f32), cnt = at::empty({E}, i64);
  at::Tensor stats = at::empty({MOE_STATS_HEAD + E}, f32), aux = at::empty({}, f32), z = at::empty({}, f32);
  const hipStream_t s = stream_of(x);
  const int xdt = code_of(x), wdt = code_of(gw);
  const size_t nbytes = moe_router_fwd_workspace(N, H, E, k, xdt, wdt);
  const FwdWorkspace ws(nbytes, x.device(), s);
  check_rc(moe_router_fwd(x.data_ptr(), xdt, gw.data_ptr(), wdt, static_cast<const float*>(ptr(bias)), N, H, E, k,
                          idx.data_ptr<int64_t>(), w.data_ptr(), w_bf16 ? MOE_BF16 : MOE_F32, logits.data_ptr<float>(),
                          lse.data_ptr<float>(), cnt.data_ptr<int64_t>(), stats.data_ptr<float>(), (float)aux_coef,
                          (float)z_coef, aux.data_ptr<float>(), z.data_ptr<float>(), ws.data_ptr(), nbytes, s),
           "moe_router_fwd");
  return {idx, w, logits, lse, cnt, stats, aux, z};
}

std::vector<at::Tensor> op_rmsnorm_router_forward(const at::Tensor& x_in, const at::Tensor& weight_in, double eps,
                                                  const at::Tensor& gw_in, int64_t k, const OptTensor& bias,
                                                  double aux_coef, double z_coef) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x_in.device());
  const at::Tensor x = x_in.contiguous(), weight = weight_in.contiguous(), gw = gw_in.contiguous();
  const int64_t N = x.size(0), H = x.size(1), E = gw.size(1);
  const auto f32 = x.options().dtype(at::kFloat);
  const auto i64 = x.options().dtype(at::kLong);
  at::Tensor xn = at::empty_like(x), rstd = at::empty({N}, f32), idx = at::empty({N, k}, i64);
  at::Tensor w = at::empty({N, k}, x.options()), logits = at::empty({N, E}, f32), lse = at::empty({N}, f32);
  at::Tensor cnt = at::empty({E}, i64), stats = at::empty({MOE_STATS_HEAD + E}, f32);
  at::Tensor aux = at::empty({}, f32), z = at::empty({}, f32);
  const hipStream_t s = stream_of(x);
  const int xdt = code_of(x), wdt = code_of(gw);
  const size_t nbytes = moe_rmsnorm_router_fwd_workspace(N, H, E, k, xdt, wdt);
  const FwdWorkspace ws(nbytes, x.device(), s);
  check_rc(moe_rmsnorm_router_fwd(x.data_ptr(), xdt, weight.data_ptr(), code_of(weight), (float)eps, gw.data_ptr(), wdt,
                                  static_cast<const float*>(ptr(bias)), N, H, E, k, xn.data_ptr(), rstd.data_ptr<float>(),
                                  idx.data_ptr<int64_t>(), w.data_ptr(), xdt, logits.data_ptr<float>(),
                                  lse.data_ptr<float>(), cnt.data_ptr<int64_t>(), stats.data_ptr<float>(),
                                  (float)aux_coef, (float)z_coef, aux.data_ptr<float>(), z.data_ptr<float>(),
                                  ws.data_ptr(), nbytes, s),
           "moe_rmsnorm_router_fwd");
  return {xn, rstd, idx, w, logits, lse, cnt, stats, aux, z};
}

std::vector<at::Tensor> op_rmsnorm_router_backward(const at::Tensor& x_in, const at::Tensor& weight_in,
                                                   const at::Tensor& rstd, const at::Tensor& xn_in, const at::Tensor& gw_in,
                                                   const at::Tensor& logits_in, const at::Tensor& idx_in,
                                                   const OptTensor& grad_w, const OptTensor& dxn, const OptTensor& cnt,
                                                   const OptTensor& grad_aux, const OptTensor& grad_z, double aux_coef,
                                                   double z_coef) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x_in.device());
  const at::Tensor x = x_in.contiguous(), weight = weight_in.contiguous(), xn = xn_in.contiguous();
  const at::Tensor gw = gw_in.contiguous(), logits = logits_in.contiguous(), idx = idx_in.contiguous();
  const int64_t N = x.size(0), H = x.size(1), E = gw.size(1), K = idx.size(1);
  at::Tensor dx = at::empty_like(x), dweight = at::empty_like(weight), dgate = at::empty({H, E}, gw.options());
  const int xdt = code_of(x), wdt = code_of(gw);
  const size_t nbytes = moe_rmsnorm_router_bwd_workspace(N, H, E, K, xdt, wdt);
  const at::Tensor ws = scratch(nbytes, x);
  check_rc(moe_rmsnorm_router_bwd(
               x.data_ptr(), xdt, weight.data_ptr(), code_of(weight), rstd.data_ptr<float>(), xn.data_ptr(), gw.data_ptr(),
               wdt, logits.data_ptr<float>(), idx.data_ptr<int64_t>(), ptr(grad_w),
               grad_w.has_value() && grad_w->defined() ? code_of(*grad_w) : MOE_F32, static_cast<const int64_t*>(ptr(cnt)),
               static_cast<const float*>(ptr(grad_aux)), static_cast<const float*>(ptr(grad_z)), (float)aux_coef,
               (float)z_coef, ptr(dxn), N, H, E, K, dx.data_ptr(), dweight.data_ptr(), dgate.data_ptr(), ws.data_ptr(),
               nbytes, stream_of(x)),
           "moe_rmsnorm_router_bwd");
  return {dx, dweight, dgate};
}

std::tuple<OptTensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor> op_plan(const at::Tensor& idx_in, int64_t E,
                                                                               int64_t capacity, int64_t layout) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(idx_in.device());
  at::Tensor idx = idx_in.contiguous();
  if (idx.scalar_type() != at::kLong) idx = idx.to(at::kLong);
  const int64_t N = idx.size(0), K = idx.size(1), M = N * K;
  const auto i32 = idx.options().dtype(at::kInt);
  OptTensor drop;
  if (capacity >= 0) drop = at::empty({N, K}, idx.options().dtype(at::kBool));
  at::Tensor row_slot = at::empty({M}, i32), slot_row = at::empty({M}, i32), offsets = at::empty({E + 1}, i32);
  at::Tensor ndrop = at::empty({1}, i32);
  const size_t nbytes = moe_plan_workspace(N, K, E);
  const at::Tensor ws = scratch(nbytes, idx);
  check_rc(moe_plan(idx.data_ptr<int64_t>(), N, K, E, capacity, (int)layout,
                    static_cast<uint8_t*>(const_cast<void*>(ptr(drop))), row_slot.data_ptr<int>(),
                    slot_row.data_ptr<int>(), offsets.data_ptr<int>(), ndrop.data_ptr<int>(), ws.data_ptr(), nbytes,
                    stream_of(idx)),
           "moe_plan");
  return {drop, row_slot, slot_row, offsets, ndrop};
}

at::Tensor op_permute(const at::Tensor& x_in, const at::Tensor& slot_row, const at::Tensor& offsets, int64_t N, int64_t K,
                      int64_t E) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x_in.device());
  const at::Tensor x = x_in.contiguous();
  const int64_t H = x.size(1);
  at::Tensor xp = at::empty({N * K, H}, x.options());
  check_rc(moe_permute(x.data_ptr(), H * x.element_size(), slot_row.data_ptr<int>(), offsets.data_ptr<int>(), N, K, E,
                       xp.data_ptr(), stream_of(x)),
           "moe_permute");
  return xp;
}

at::Tensor op_combine(const at::Tensor& y_in, const at::Tensor& w_in, const OptTensor& drop, const at::Tensor& slot_row,
                      const at::Tensor& offsets, int64_t N, int64_t K, int64_t E) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(y_in.device());
  const at::Tensor y = y_in.contiguous(), w = w_in.contiguous();
  const int64_t H = y.size(1);
  at::Tensor out = at::empty({N, H}, y.options());
  check_rc(moe_combine(y.data_ptr(), code_of(y), w.data_ptr(), code_of(w), static_cast<const uint8_t*>(ptr(drop)),
                       slot_row.data_ptr<int>(), offsets.data_ptr<int>(), N, K, H, E, out.data_ptr(), stream_of(y)),
           "moe_combine");
  return out;
}

std::tuple<at::Tensor, OptTensor> op_combine_backward(const at::Tensor& dout_in, const at::Tensor& y, const at::Tensor& w_in,
                                                      const OptTensor& drop, const at::Tensor& slot_row,
                                                      const at::Tensor& offsets, int64_t N, int64_t K, int64_t E,
                                                      bool need_dw, bool zero_tail) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(y.device());
  const at::Tensor dout = dout_in.contiguous(), w = w_in.contiguous();
  const int64_t H = y.size(1);
  at::Tensor dy = at::empty_like(y);
  OptTensor dw;
  if (need_dw) dw = at::empty({N, K}, w.options());
  const hipStream_t s = stream_of(y);
  check_rc(moe_combine_bwd(dout.data_ptr(), y.data_ptr(), code_of(y), w.data_ptr(), code_of(w),
                           static_cast<const uint8_t*>(ptr(drop)), slot_row.data_ptr<int>(), offsets.data_ptr<int>(), N, K,
                           H, E, dy.data_ptr(), const_cast<void*>(ptr(dw)), s),
           "moe_combine_bwd");
  if (zero_tail)
    check_rc(moe_zero_tail(dy.data_ptr(), H * dy.element_size(), offsets.data_ptr<int>(), E, dy.size(0), s),
             "moe_zero_tail");
  return {dy, dw};
}

at::Tensor op_unpermute_sum(const at::Tensor& dxp_in, const OptTensor& addend_in, const at::Tensor& slot_row,
                            const at::Tensor& offsets, int64_t N, int64_t K, int64_t E) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(dxp_in.device());
  const at::Tensor dxp = dxp_in.contiguous();
  OptTensor addend;
  if (addend_in.has_value() && addend_in->defined()) addend = addend_in->contiguous();
  const int64_t H = dxp.size(1);
  at::Tensor dx = at::empty({N, H}, dxp.options());
  check_rc(moe_unpermute_sum(dxp.data_ptr(), ptr(addend), code_of(dxp), slot_row.data_ptr<int>(), offsets.data_ptr<int>(),
                             N, K, H, E, dx.data_ptr(), stream_of(dxp)),
           "moe_unpermute_sum");
  return dx;
}

// Bytes of the grouped GEMM's tile tables and of the partial tiles of products split over k.
size_t gemm_workspace(bool f32, bool fwd, int64_t R, int64_t H, int64_t F, int64_t E) {
  if (f32)
    return moe_swiglu_f32_workspace(E) +
           (fwd ? moe_swiglu_fwd_f32_split_workspace(R, H, F, E) : moe_swiglu_f32_split_workspace(R, H, F, E));
  return moe_swiglu_workspace(E) +
         (fwd ? moe_swiglu_fwd_split_workspace(R, H, F, E) : moe_swiglu_split_workspace(R, H, F, E));
}

std::tuple<at::Tensor, OptTensor, at::Tensor> op_swiglu_forward(const at::Tensor& xp, const at::Tensor& wg,
                                                                const at::Tensor& wu, const at::Tensor& wd,
                                                                const at::Tensor& offsets, bool keep_preact) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(xp.device());
  const bool f32 = xp.scalar_type() == at::kFloat;
  const int64_t R = xp.size(0), H = xp.size(1), E = wg.size(0), F = wg.size(1);
  at::Tensor act = at::empty({R, F}, xp.options()), y = at::empty({R, H}, xp.options());
  OptTensor hgu;
  if (keep_preact) hgu = at::empty({R, 2 * F}, xp.options());
  const size_t nbytes = gemm_workspace(f32, true, R, H, F, E);
  const at::Tensor ws = scratch(nbytes, xp);
  const hipStream_t s = stream_of(xp);
  void* const h = const_cast<void*>(ptr(hgu));
  if (f32)
    check_rc(moe_swiglu_fwd_f32(xp.data_ptr<float>(), wg.data_ptr<float>(), wu.data_ptr<float>(), wd.data_ptr<float>(),
                                offsets.data_ptr<int>(), R, H, F, E, act.data_ptr<float>(), static_cast<float*>(h),
                                y.data_ptr<float>(), ws.data_ptr(), nbytes, s),
             "moe_swiglu_fwd_f32");
  else
    check_rc(moe_swiglu_fwd(xp.data_ptr(), wg.data_ptr(), wu.data_ptr(), wd.data_ptr(), offsets.data_ptr<int>(), R, H, F, E,
                            act.data_ptr(), h, y.data_ptr(), ws.data_ptr(), nbytes, s),
             "moe_swiglu_fwd");
  return {act, hgu, y};
}

std::vector<at::Tensor> op_swiglu_backward(const at::Tensor& dy, const at::Tensor& xp, const at::Tensor& act,
                                           const at::Tensor& hgu, const at::Tensor& wg, const at::Tensor& wu,
                                           const at::Tensor& wd, const at::Tensor& offsets) {
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(xp.device());
  const bool f32 = xp.scalar_type() == at::kFloat;
  const int64_t R = xp.size(0), H = xp.size(1), E = wg.size(0), F = wg.size(1);
  at::Tensor dh = at::empty({R, 2 * F}, xp.options()), dxp = at::empty({R, H}, xp.options());
  at::Tensor dwg = at::empty_like(wg), dwu = at::empty_like(wu), dwd = at::empty_like(wd);
  const size_t nbytes = gemm_workspace(f32, false, R, H, F, E);
  const at::Tensor ws = scratch(nbytes, xp);
  const hipStream_t s = stream_of(xp);
  if (f32)
    check_rc(moe_swiglu_bwd_f32(dy.data_ptr<float>(), xp.data_ptr<float>(), act.data_ptr<float>(), hgu.data_ptr<float>(),
                                wg.data_ptr<float>(), wu.data_ptr<float>(), wd.data_ptr<float>(), offsets.data_ptr<int>(), R,
                                H, F, E, dh.data_ptr<float>(), dxp.data_ptr<float>(), dwg.data_ptr<float>(),
                                dwu.data_ptr<float>(), dwd.data_ptr<float>(), ws.data_ptr(), nbytes, s),
             "moe_swiglu_bwd_f32");
  else
    check_rc(moe_swiglu_bwd(dy.data_ptr(), xp.data_ptr(), act.data_ptr(), hgu.data_ptr(), wg.data_ptr(), wu.data_ptr(),
                            wd.data_ptr(), offsets.data_ptr<int>(), R, H, F, E, dh.data_ptr(), dxp.data_ptr(),
                            dwg.data_ptr(), dwu.data_ptr(), dwd.data_ptr(), ws.data_ptr(), nbytes, s),
             "moe_swiglu_bwd");
  return {dxp, dwg, dwu, dwd};
}

}  // namespace

PYBIND11_MODULE(_moe_torch, m) {
  m.doc() = "Native autograd binding of the fused HIP router (forward and backward over the moe_mi355 C ABI).";
  // No call holds the GIL: none touches a Python object, and one that waits (for the allocator, a full queue or the
  // workspace lock) holds up no other thread.
  const pybind11::call_guard<pybind11::gil_scoped_release> nogil;
  m.def("router_core", &router_core, "(x, gate_w, k, aux_coef, z_coef, bias) -> (idx, w, aux, z, logits, cnt, stats)",
        pybind11::arg("x"), pybind11::arg("gate_w"), pybind11::arg("k"), pybind11::arg("aux_coef"),
        pybind11::arg("z_coef"), pybind11::arg("bias") = pybind11::none(), pybind11::arg("link_x") = false, nogil);
  m.def("router_forward", &op_router_forward, nogil);
  m.def("rmsnorm_router_forward", &op_rmsnorm_router_forward, nogil);
  m.def("rmsnorm_router_backward", &op_rmsnorm_router_backward, nogil);
  m.def("plan", &op_plan, nogil);
  m.def("permute", &op_permute, nogil);
  m.def("combine", &op_combine, nogil);
  m.def("combine_backward", &op_combine_backward, nogil);
  m.def("unpermute_sum", &op_unpermute_sum, nogil);
  m.def("swiglu_forward", &op_swiglu_forward, nogil);
  m.def("swiglu_backward", &op_swiglu_backward, nogil);
}

// block_host.cpp — host side of the MoE block's forward and backward: output
// allocation and the launch sequence over the C ABI, as one call each.
//
// The same sequence through the Python wrappers of fusionllm_amd/_kernels.py
// (one ctypes call, its argument checks and one torch.empty per output at a
// time) took 115 us of host time for a forward and 200 us for a backward pass
// at 8 experts, longer than the kernels of up to about 2000 tokens; here 74 and
// 127 us with what autograd's Function around them costs (a training pass of
// 1021 tokens, host-bound, 555 -> 440 us).  The wrappers remain the public way
// to call one entry point, and the block's path while per-entry-point timing
// is on.
//
// Reference: FusionLLM models/moe.py:79-87 (forward) and its autograd.
#include <torch/extension.h>

#include <algorithm>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/fusionmoe.h"

namespace {

using at::Tensor;

// The entry points of the library that fusionllm_amd._lib loaded (bind), so
// that a program which chose another build of it launches that one here too.
#define FMOE_ENTRY_POINTS(F)                                                                              \
  F(fmoe_status_string) F(fmoe_split_workspace_bytes) F(fmoe_route_and_dispatch_workspace_bytes)          \
  F(fmoe_route_and_dispatch) F(fmoe_gateup_fwd) F(fmoe_down_fwd) F(fmoe_combine_fwd) F(fmoe_combine_bwd)  \
  F(fmoe_down_bwd_dx) F(fmoe_weight_grad_workspace_bytes) F(fmoe_weight_grad) F(fmoe_gateup_bwd_dx)       \
  F(fmoe_router_bwd_workspace_bytes) F(fmoe_router_bwd)
struct Api {
#define F(name) decltype(&::name) name = nullptr;
  FMOE_ENTRY_POINTS(F)
#undef F
} api;

// Names of the entry points used here.
std::vector<std::string> entry_points() {
#define F(name) #name,
  return {FMOE_ENTRY_POINTS(F)};
#undef F
}

// Their addresses, in that order.
void bind(const std::vector<uint64_t>& addresses) {
  if (addresses.size() != entry_points().size()) throw std::runtime_error("one address per entry point is needed");
  size_t i = 0;
#define F(name) api.name = reinterpret_cast<decltype(api.name)>(addresses[i++]);
  FMOE_ENTRY_POINTS(F)
#undef F
}

void need_entry_points() {
  if (api.fmoe_status_string == nullptr) throw std::runtime_error("bind() has not been called");
}

// A status other than FMOE_OK; becomes fusionllm_amd._lib.FusionMoEError in Python.
struct StatusError : std::runtime_error {
  using std::runtime_error::runtime_error;
};
[[noreturn]] void raise_status(int rc, const char* what) {
  throw StatusError(std::string(what) + " failed: " + api.fmoe_status_string(rc) + " (status " + std::to_string(rc) + ")");
}
void check(int rc, const char* what) {
  if (rc != FMOE_OK) raise_status(rc, what);
}

// Address of a contiguous device tensor of the given dtype.
void* req(const Tensor& t, const char* name, at::ScalarType dtype) {
  if (!t.is_cuda()) throw std::runtime_error(std::string(name) + " must be a ROCm device tensor");
  if (!t.is_contiguous()) throw std::runtime_error(std::string(name) + " must be contiguous");
  if (t.scalar_type() != dtype)
    throw std::runtime_error(std::string(name) + " must be " + c10::toString(dtype) + " (got " +
                             c10::toString(t.scalar_type()) + ")");
  return t.data_ptr();
}

int dtype_code(at::ScalarType t) {
  if (t == at::kBFloat16) return FMOE_BF16;
  if (t == at::kFloat) return FMOE_F32;
  throw std::runtime_error(std::string("unsupported dtype ") + c10::toString(t));
}

Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, const Tensor& like) {
  return at::empty(shape, like.options().dtype(dtype).requires_grad(false));
}

// The dtype in which one launch writes gradients of the dtypes own: theirs if they share it, else
// fp32, from which each is rounded to its own (the kernel writes every group in one dtype).
at::ScalarType launch_dtype(const std::vector<at::ScalarType>& own) {
  for (const at::ScalarType t : own)
    if (t != own[0]) return at::kFloat;
  return own[0];
}

// Addresses of the groups' weights, each checked against its shape.
std::vector<const void*> weight_ptrs(const std::vector<Tensor>& ws, size_t G, const char* name, int64_t rows,
                                     int64_t cols) {
  if (ws.size() < G)
    throw std::runtime_error("needs " + std::to_string(G) + " " + name + " matrices (got " +
                             std::to_string(ws.size()) + ")");
  std::vector<const void*> p(G);
  for (size_t g = 0; g < G; ++g) {
    p[g] = req(ws[g], name, at::kBFloat16);
    if (ws[g].dim() != 2 || ws[g].size(0) != rows || ws[g].size(1) != cols)
      throw std::runtime_error(std::string(name) + " must be (" + std::to_string(rows) + ", " +
                               std::to_string(cols) + ")");
  }
  return p;
}

// Bytes of split workspace that a row product of K steps k_steps and tile_cols
// output tiles per 256-row block can use: none if it runs every tile whole (as
// _split_workspace of _kernels.py, and launch_rows of the library, have it):
// fewer than 16 steps, 8 full rounds of tiles or more, or a forward launch
// (small) whose groups all go to the small-group kernel.
size_t split_bytes(int64_t rows_routed, int64_t rows_shared, int64_t k_steps, int64_t tile_cols, bool small) {
  if (k_steps < 16) return 0;
  if (small && rows_routed <= 256 && rows_shared <= 128 && rows_routed + rows_shared <= 4096) return 0;
  const size_t bytes = api.fmoe_split_workspace_bytes();
  const int64_t cus = static_cast<int64_t>(bytes / (256 * 256 * sizeof(float)));  // one partial tile per CU
  const int64_t blocks = (rows_routed + 255) / 256 + (rows_shared + 255) / 256;
  return blocks * tile_cols >= 8 * cus ? 0 : bytes;
}

// One workspace for a pass: its launches run one after the other on one
// stream, so the largest request serves all of them.
struct Workspace {
  Tensor buf;
  size_t bytes;
  Workspace(size_t n, const Tensor& like) : bytes(n) {
    if (n) buf = empty({static_cast<int64_t>(n)}, at::kByte, like);
  }
  void* ptr() const { return bytes ? buf.data_ptr() : nullptr; }
};

// Routing, dispatch, gate/up, down and combine (more than 128 tokens, dim <=
// 2048).  Returns idx, idx64, w, v, counts, offsets, perm, pos, x_perm, ab, h,
// o, y.
std::vector<Tensor> forward(const Tensor& x, const Tensor& gate_w, const Tensor& gate_b,
                            const std::vector<Tensor>& w1, const std::vector<Tensor>& w3,
                            const std::vector<Tensor>& w2, int64_t k, int64_t inter, double route_scale,
                            bool has_shared, at::ScalarType out_dtype, const c10::optional<Tensor>& residual,
                            const c10::optional<Tensor>& counts_host, uint64_t stream) {
  need_entry_points();
  void* s = reinterpret_cast<void*>(stream);
  const int64_t T = x.size(0), d = x.size(1);
  const int E = static_cast<int>(gate_w.size(0));
  const size_t G = static_cast<size_t>(E) + (has_shared ? 1 : 0);
  const int64_t rows_r = T * k, rows_s = has_shared ? T : 0, rows = rows_r + rows_s;
  const int kk = static_cast<int>(k);
  const auto bf = at::kBFloat16;
  const void *xp = req(x, "x", bf), *gwp = req(gate_w, "gate.weight", bf), *gbp = req(gate_b, "gate.bias", bf);
  const auto p1 = weight_ptrs(w1, G, "w1", inter, d), p3 = weight_ptrs(w3, G, "w3", inter, d),
             p2 = weight_ptrs(w2, G, "w2", d, inter);
  Tensor idx = empty({T, k}, at::kInt, x), idx64 = empty({T, k}, at::kLong, x), w = empty({T, k}, at::kFloat, x),
         v = empty({T, k}, at::kFloat, x), counts = empty({E}, at::kInt, x), offsets = empty({E + 1}, at::kInt, x),
         perm = empty({rows_r}, at::kInt, x), pos = empty({rows_r}, at::kInt, x), x_perm = empty({rows_r, d}, bf, x);
  void* ch = nullptr;
  if (counts_host.has_value()) {
    const Tensor& c = *counts_host;
    if (c.is_cuda() || c.scalar_type() != at::kInt || c.numel() < E || !c.is_contiguous() || !c.is_pinned())
      throw std::runtime_error("counts_host must be a contiguous pinned int32 CPU tensor of n_experts elements");
    ch = c.data_ptr();
  }
  const size_t split = std::max(split_bytes(rows_r, rows_s, d / 64, (inter + 127) / 128, true),
                                split_bytes(rows_r, rows_s, inter / 64, (d + 255) / 256, true));
  const size_t rd = api.fmoe_route_and_dispatch_workspace_bytes(T, E, kk);
  const Workspace ws(std::max(split, rd), x);
  check(api.fmoe_route_and_dispatch(xp, gwp, gbp, T, d, E, kk, static_cast<float>(route_scale),
                                static_cast<int32_t*>(idx.data_ptr()), static_cast<int64_t*>(idx64.data_ptr()),
                                static_cast<float*>(w.data_ptr()), static_cast<float*>(v.data_ptr()),
                                static_cast<int32_t*>(counts.data_ptr()), static_cast<int32_t*>(offsets.data_ptr()),
                                static_cast<int32_t*>(perm.data_ptr()), static_cast<int32_t*>(pos.data_ptr()),
                                x_perm.data_ptr(), static_cast<int32_t*>(ch), ws.ptr(), rd, s),
        "fmoe_route_and_dispatch");
  const int32_t* off = static_cast<const int32_t*>(offsets.data_ptr());
  Tensor ab = empty({rows, 2 * inter}, bf, x), h = empty({rows, inter}, bf, x);
  check(api.fmoe_gateup_fwd(x_perm.data_ptr(), nullptr, kk, rows_r, has_shared ? xp : nullptr, off, E, rows_r, rows_s, d,
                        inter, p1.data(), p3.data(), ab.data_ptr(), h.data_ptr(), ws.ptr(), split, s),
        "fmoe_gateup_fwd");
  Tensor o = empty({rows, d}, bf, x);
  check(api.fmoe_down_fwd(h.data_ptr(), off, E, rows_r, rows_s, d, inter, p2.data(), o.data_ptr(), ws.ptr(), split, s),
        "fmoe_down_fwd");
  Tensor y = empty({T, d}, out_dtype, x);
  const void* res = residual.has_value() ? req(*residual, "residual", out_dtype) : nullptr;
  check(api.fmoe_combine_fwd(o.data_ptr(), static_cast<int32_t*>(idx.data_ptr()), static_cast<float*>(w.data_ptr()),
                         static_cast<int32_t*>(pos.data_ptr()), T, d, kk, rows_r, has_shared, dtype_code(out_dtype),
                         res, y.data_ptr(), s),
        "fmoe_combine_fwd");
  return {idx, idx64, w, v, counts, offsets, perm, pos, x_perm, ab, h, o, y};
}

// Combine backward, down dX, dW2, gate/up dX, dW1|dW3 and the router's
// backward.  Returns dx_rows, d_logits, d gate.weight, d gate.bias (in the
// gate weight's gradient dtype), then dw1, dw3, dw2 of every group in turn.
std::vector<Tensor> backward(const Tensor& dy, const Tensor& x, const Tensor& gate_w, const Tensor& w,
                             const Tensor& v, const Tensor& offsets, const Tensor& perm, const Tensor& x_perm,
                             const Tensor& ab, const Tensor& h, const Tensor& o, const std::vector<Tensor>& w1,
                             const std::vector<Tensor>& w3, const std::vector<Tensor>& w2, int64_t k, int64_t inter,
                             double route_scale, bool has_shared, at::ScalarType gate_grad_dtype,
                             const std::vector<at::ScalarType>& grad_dtypes, uint64_t stream) {
  need_entry_points();
  void* s = reinterpret_cast<void*>(stream);
  const int64_t T = x.size(0), d = x.size(1);
  const int E = static_cast<int>(gate_w.size(0));
  const size_t G = static_cast<size_t>(E) + (has_shared ? 1 : 0);
  const int64_t rows_r = T * k, rows_s = has_shared ? T : 0, rows = rows_r + rows_s;
  const int kk = static_cast<int>(k);
  const float rs = static_cast<float>(route_scale);
  const auto bf = at::kBFloat16;
  const auto p1 = weight_ptrs(w1, G, "w1", inter, d), p3 = weight_ptrs(w3, G, "w3", inter, d),
             p2 = weight_ptrs(w2, G, "w2", d, inter);
  const void *dyp = req(dy, "dy", dy.scalar_type()), *xp = req(x, "x", bf), *op = req(o, "expert_out", bf),
             *wp = req(w, "weights", at::kFloat), *pp = req(perm, "perm", at::kInt),
             *offp = req(offsets, "offsets", at::kInt), *abp = req(ab, "ab", bf), *hp = req(h, "h", bf),
             *xpp = req(x_perm, "x_perm", bf), *vp = req(v, "topv", at::kFloat);
  const int32_t* off = static_cast<const int32_t*>(offp);
  const int32_t* permp = static_cast<const int32_t*>(pp);
  const size_t split = std::max(split_bytes(rows_r, rows_s, d / 64, (inter + 255) / 256, false),
                                split_bytes(rows_r, rows_s, 2 * inter / 64, (d + 255) / 256, false));
  const size_t g2 = api.fmoe_weight_grad_workspace_bytes(rows_r, rows_s, E, d, inter);
  const size_t g13 = api.fmoe_weight_grad_workspace_bytes(rows_r, rows_s, E, 2 * inter, d);
  const size_t rb = api.fmoe_router_bwd_workspace_bytes(T, d, E, kk);
  const Workspace ws(std::max(std::max(split, rb), std::max(g2, g13)), x);

  Tensor d_o = empty({rows_r, d}, bf, x), d_w = empty({T, k}, at::kFloat, x);
  check(api.fmoe_combine_bwd(dyp, dtype_code(dy.scalar_type()), op, static_cast<const float*>(wp), permp, T, d, kk,
                         d_o.data_ptr(), static_cast<float*>(d_w.data_ptr()), s),
        "fmoe_combine_bwd");
  Tensor dy_sh = has_shared ? dy.to(bf).contiguous() : Tensor();
  const void* dsp = has_shared ? dy_sh.data_ptr() : nullptr;
  Tensor d_ab = empty({rows, 2 * inter}, bf, x);
  check(api.fmoe_down_bwd_dx(d_o.data_ptr(), dsp, off, E, rows_r, rows_s, d, inter, p2.data(), abp, d_ab.data_ptr(),
                         ws.ptr(), split, s),
        "fmoe_down_bwd_dx");

  std::vector<at::ScalarType> t13, t2;
  for (size_t g = 0; g < G; ++g) {
    t13.push_back(grad_dtypes.at(3 * g));
    t13.push_back(grad_dtypes.at(3 * g + 1));
    t2.push_back(grad_dtypes.at(3 * g + 2));
  }
  const at::ScalarType dt13 = launch_dtype(t13), dt2 = launch_dtype(t2);
  std::vector<Tensor> out(4 + 3 * G);
  std::vector<void*> o1(G), o3(G), o2(G);
  for (size_t g = 0; g < G; ++g) {
    out[4 + 3 * g] = empty({inter, d}, dt13, x);
    out[5 + 3 * g] = empty({inter, d}, dt13, x);
    out[6 + 3 * g] = empty({d, inter}, dt2, x);
    o1[g] = out[4 + 3 * g].data_ptr();
    o3[g] = out[5 + 3 * g].data_ptr();
    o2[g] = out[6 + 3 * g].data_ptr();
  }
  check(api.fmoe_weight_grad(d_o.data_ptr(), dsp, d, hp, nullptr, inter, nullptr, 1, rows, off, E, rows_r, rows_s, d,
                         inter, d, o2.data(), nullptr, dtype_code(dt2), ws.ptr(), g2, s),
        "fmoe_weight_grad");
  out[0] = empty({rows, d}, bf, x);
  check(api.fmoe_gateup_bwd_dx(d_ab.data_ptr(), off, E, rows_r, rows_s, d, inter, p1.data(), p3.data(),
                           out[0].data_ptr(), ws.ptr(), split, s),
        "fmoe_gateup_bwd_dx");
  check(api.fmoe_weight_grad(d_ab.data_ptr(), nullptr, 2 * inter, xpp, has_shared ? xp : nullptr, d, nullptr, 1, rows_r,
                         off, E, rows_r, rows_s, 2 * inter, d, inter, o1.data(), o3.data(),
                         dtype_code(dt13), ws.ptr(), g13, s),
        "fmoe_weight_grad");
  out[1] = empty({T, k}, at::kFloat, x);
  out[2] = empty({E, d}, gate_grad_dtype, x);
  out[3] = empty({E}, gate_grad_dtype, x);
  check(api.fmoe_router_bwd(static_cast<const float*>(d_w.data_ptr()), static_cast<const float*>(vp), permp, off, xp, T,
                        d, E, kk, rs, static_cast<float*>(out[1].data_ptr()), out[2].data_ptr(), out[3].data_ptr(),
                        dtype_code(gate_grad_dtype), ws.ptr(), rb, s),
        "fmoe_router_bwd");
  for (size_t i = 0; i < 3 * G; ++i)
    if (out[4 + i].scalar_type() != grad_dtypes[i]) out[4 + i] = out[4 + i].to(grad_dtypes[i]);
  return out;
}

}  // namespace

// Other Python threads run during a sequence, as they do during a ctypes call.
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::register_local_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const StatusError& e) {
      PyErr_SetString(py::object(py::module_::import("fusionllm_amd._lib").attr("FusionMoEError")).ptr(), e.what());
    }
  });
  m.def("entry_points", &entry_points);
  m.def("bind", &bind);
  m.def("forward", &forward, py::call_guard<py::gil_scoped_release>());
  m.def("backward", &backward, py::call_guard<py::gil_scoped_release>());
}

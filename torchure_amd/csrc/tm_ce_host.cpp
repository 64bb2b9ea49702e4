// tm_ce_host.cpp -- host side of one fused linear + cross-entropy call (CPU code only).
//
// A call issues 4 to 5 kernels per chunk of rows, with a buffer for each result. Driven from
// Python (a foreign-function call of 8 to 12 arguments and one or two allocations for every
// kernel) that took 70 us a call on the host before the GPU work of a small head (512 x 256 x
// 4096: 60 us) could hide it; this loop takes 25. It holds no state between calls but the entry
// points' addresses, and decides nothing about shapes: the caller passes each chunk's padding and
// choice of product. Every kernel is reached through the C ABI (include/torchure_amd.h).

#include <torch/extension.h>
#include <torch/csrc/Exceptions.h>

#include <cstdint>
#include <string>
#include <vector>

namespace py = pybind11;

namespace {

using i64 = int64_t;
typedef int (*cast2_t)(void*, const void*, i64, void*, const void*, i64, void*);
typedef int (*logits_t)(void*, i64, const void*, const void*, i64, i64, i64, void*);
typedef int (*rows_t)(void*, i64, const void*, i64, i64, i64, i64, void*, void*);
typedef int (*rows_loss_t)(const void*, i64, const void*, i64, i64, i64, void*, void*);
typedef size_t (*gh_bytes_t)(i64, i64, i64);
typedef int (*grad_h_t)(void*, const void*, i64, const void*, i64, i64, i64, void*, size_t, void*);
typedef int (*grad_w_t)(void*, const void*, i64, i64, const void*, i64, i64, i64, void*, size_t, void*);
typedef int (*fold_t)(void*, const void* const*, int, i64, int, const void*, const void*, void*);
typedef int (*mean_t)(const void*, const void*, i64, i64, void*, void*, void*);
typedef int (*finish_t)(void*, const void* const*, int, i64, int, const void*, void*, i64, int, const void*, const void*,
                        void*);
typedef const char* (*error_t)();

struct Abi {
  cast2_t cast2;
  logits_t logits;
  rows_t rows;
  rows_loss_t rows_loss;
  gh_bytes_t grad_h_bytes, grad_w_bytes;
  grad_h_t grad_h;
  grad_w_t grad_w;
  fold_t fold;
  mean_t mean_loss;
  finish_t finish;
  error_t last_error;
  py::object native_error;
};
Abi* g_abi = nullptr;  // set once, at the first call, under the GIL

void ce_bind(const py::dict& addresses, const py::object& native_error) {
  if (g_abi) return;
  auto at = [&](const char* name) { return reinterpret_cast<void*>(addresses[name].cast<uintptr_t>()); };
  Abi* a = new Abi();
  a->cast2 = reinterpret_cast<cast2_t>(at("tm_ce_cast2"));
  a->logits = reinterpret_cast<logits_t>(at("tm_ce_logits_ld_bf16"));
  a->rows = reinterpret_cast<rows_t>(at("tm_ce_rows_padded_bf16"));
  a->rows_loss = reinterpret_cast<rows_loss_t>(at("tm_ce_rows_loss_bf16"));
  a->grad_h_bytes = reinterpret_cast<gh_bytes_t>(at("tm_ce_grad_h_ld_workspace_bytes"));
  a->grad_w_bytes = reinterpret_cast<gh_bytes_t>(at("tm_ce_grad_w_ld_workspace_bytes"));
  a->grad_h = reinterpret_cast<grad_h_t>(at("tm_ce_grad_h_ld_bf16"));
  a->grad_w = reinterpret_cast<grad_w_t>(at("tm_ce_grad_w_ld_bf16"));
  a->fold = reinterpret_cast<fold_t>(at("tm_ce_grad_w_fold"));
  a->mean_loss = reinterpret_cast<mean_t>(at("tm_ce_mean_loss"));
  a->finish = reinterpret_cast<finish_t>(at("tm_ce_finish"));
  a->last_error = reinterpret_cast<error_t>(at("tm_last_error"));
  a->native_error = native_error;
  g_abi = a;
}

const Abi& abi() {
  if (!g_abi) throw std::runtime_error("torchure_amd._tm_host: ce_bind was not called");
  return *g_abi;
}

struct EntryFailed : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check(int rc, const char* what) {
  if (rc != 0)
    throw EntryFailed(std::string(what) + " failed (" + std::to_string(rc) + "): " + abi().last_error());
}

// Runs body without the GIL: its allocations may wait for the device, and its launches for room in
// the queue, while other Python threads go on. A failed entry point becomes
// torchure_amd._native.NativeError, as from the Python callers.
template <typename Body>
auto without_gil(Body&& body) -> decltype(body()) {
  try {
    py::gil_scoped_release released;
    return body();
  } catch (const EntryFailed& e) {  // the GIL is held again
    PyErr_SetString(abi().native_error.ptr(), e.what());
    throw py::error_already_set();
  }
}

char* ptr(const at::Tensor& t) { return t.defined() ? static_cast<char*>(t.data_ptr()) : nullptr; }

py::object or_none(const at::Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

// The chunks of one call. hidden (n x d) and weight (v x d) are contiguous, bf16 or (cast_h,
// cast_w) fp32; the chunks have `chunk` rows, the last one the rest, and their logits
// pad[0] x ld (the last one's pad[1] x ld). The logits and their row pass run over `group` chunks
// at a time, in one buffer (group > 1 only where a chunk has no padding rows of its own). own_h[i]:
// grad_h on the split-K kernel, else the library's product. grad = false: the loss alone. An
// allocation that fails leaves nothing held: the caller may call again with less to hold.
struct Forward {
  at::Tensor loss, out2;  // out2: loss sum, n_valid
  at::Tensor grad_hidden, grad_weight;
  std::vector<at::Tensor> pending;  // chunks' grad_W still to be added, the last one at the end
  bool accumulated = false;         // whether grad_weight holds earlier chunks
};

Forward run_forward(const at::Tensor& hidden, const at::Tensor& weight, bool cast_h, bool cast_w,
                     const at::Tensor& labels, i64 ignore, i64 chunk, i64 group, std::pair<i64, i64> pad, i64 ld,
                     std::pair<bool, bool> own_h, bool grad, bool want_h, bool want_w, i64 fold_chunks, i64 fold_bytes,
                     uintptr_t stream_handle) {
  const Abi& a = abi();
  void* stream = reinterpret_cast<void*>(stream_handle);
  const i64 n = hidden.size(0), d = hidden.size(1), v = weight.size(0);
  const auto f32 = hidden.options().dtype(at::kFloat).requires_grad(false);
  const auto bf16 = f32.dtype(at::kBFloat16);
  at::Tensor h = cast_h ? at::empty({n, d}, bf16) : hidden, w = cast_w ? at::empty({v, d}, bf16) : weight;
  if (cast_h || cast_w)
    check(a.cast2(cast_h ? ptr(h) : nullptr, cast_h ? ptr(hidden) : nullptr, cast_h ? n * d : 0,
                  cast_w ? ptr(w) : nullptr, cast_w ? ptr(weight) : nullptr, cast_w ? v * d : 0, stream),
          "tm_ce_cast2");
  const i64 last = n - (n - 1) / chunk * chunk;  // rows of the last chunk
  at::Tensor row_loss = at::empty({n}, f32), ws;
  Forward out;
  at::Tensor &grad_hidden = out.grad_hidden, &grad_weight = out.grad_weight;
  std::vector<at::Tensor>& pending = out.pending;
  // one workspace for both gradients' split sums over the chunks (stream-ordered)
  size_t bytes = 0;
  if (grad && want_h) {
    grad_hidden = at::empty({n, d}, bf16);
    if (own_h.first && n > chunk) bytes = a.grad_h_bytes(chunk, v, d);
    if (own_h.second) bytes = std::max(bytes, a.grad_h_bytes(last, v, d));
  }
  if (grad && want_w) {
    if (n > chunk) bytes = std::max(bytes, a.grad_w_bytes(pad.first, v, d));
    bytes = std::max(bytes, a.grad_w_bytes(pad.second, v, d));
  }
  if (bytes) ws = at::empty({static_cast<i64>(bytes)}, f32.dtype(at::kByte));
  at::Tensor held;  // the group's logits
  i64 first = 0, until = 0;  // and its rows
  for (i64 s = 0; s < n; s += chunk) {
    const bool is_last = s + chunk >= n;
    const i64 rows = is_last ? last : chunk, pad_rows = grad ? (is_last ? pad.second : pad.first) : rows;
    const char* hs = ptr(h) + s * d * 2;
    if (s >= until) {
      held = at::Tensor();
      first = s;
      until = std::min(n, s + group * chunk);
      const i64 over = until == n ? (grad ? pad.second - last : 0) : pad_rows - rows;
      held = at::empty({until - s + over, ld}, bf16);
      const i64* lab = labels.data_ptr<i64>() + s;
      float* losses = row_loss.data_ptr<float>() + s;
      check(a.logits(ptr(held), ld, hs, ptr(w), until - s, v, d, stream), "tm_ce_logits_ld_bf16");
      if (grad)
        check(a.rows(ptr(held), ld, lab, until - s, held.size(0), v, ignore, losses, stream), "tm_ce_rows_padded_bf16");
      else
        check(a.rows_loss(ptr(held), ld, lab, until - s, v, ignore, losses, stream), "tm_ce_rows_loss_bf16");
    }
    if (!grad) continue;
    const at::Tensor logits = held.narrow(0, s - first, pad_rows);
    if (want_h) {
      if (is_last ? own_h.second : own_h.first) {
        check(a.grad_h(ptr(grad_hidden) + s * d * 2, ptr(logits), ld, ptr(w), rows, v, d, ptr(ws), bytes, stream),
              "tm_ce_grad_h_ld_bf16");
      } else {
        at::Tensor gh = grad_hidden.narrow(0, s, rows);
        at::mm_out(gh, logits.narrow(0, 0, rows).narrow(1, 0, v), w);
      }
    }
    if (want_w) {
      at::Tensor gw = at::empty({v, d}, bf16);
      check(a.grad_w(ptr(gw), ptr(logits), ld, pad_rows, hs, rows, v, d, ptr(ws), bytes, stream), "tm_ce_grad_w_ld_bf16");
      pending.push_back(gw);
      const i64 waiting = static_cast<i64>(pending.size());
      if (!is_last && (waiting == fold_chunks || waiting * v * d * 2 >= fold_bytes)) {
        if (!grad_weight.defined()) grad_weight = at::empty({v, d}, f32);
        std::vector<const void*> p;
        for (const at::Tensor& t : pending) p.push_back(ptr(t));
        check(a.fold(ptr(grad_weight), p.data(), static_cast<int>(waiting), v * d, out.accumulated, nullptr, nullptr,
                     stream),
              "tm_ce_grad_w_fold");
        out.accumulated = true;
        pending.clear();
      }
    }
  }
  out.out2 = at::empty({2}, f32);
  out.loss = at::empty({}, f32);
  check(a.mean_loss(ptr(row_loss), ptr(labels), n, ignore, ptr(out.out2), ptr(out.loss), stream), "tm_ce_mean_loss");
  return out;
}

// Returns (loss, out2, grad_hidden, grad_weight, pending, accumulated) of run_forward.
py::tuple ce_forward(const at::Tensor& hidden, const at::Tensor& weight, bool cast_h, bool cast_w,
                     const at::Tensor& labels, i64 ignore, i64 chunk, i64 group, std::pair<i64, i64> pad, i64 ld,
                     std::pair<bool, bool> own_h, bool grad, bool want_h, bool want_w, i64 fold_chunks, i64 fold_bytes,
                     uintptr_t stream_handle) {
  HANDLE_TH_ERRORS
  const Forward f = without_gil([&] {
    return run_forward(hidden, weight, cast_h, cast_w, labels, ignore, chunk, group, pad, ld, own_h, grad, want_h,
                       want_w, fold_chunks, fold_bytes, stream_handle);
  });
  return py::make_tuple(f.loss, f.out2, or_none(f.grad_hidden), or_none(f.grad_weight), py::cast(f.pending),
                        f.accumulated);
  END_HANDLE_TH_ERRORS_PYBIND
}

// Backward: the waiting chunks added into grad_weight (made here if there is none and want_w) and
// both gradients scaled by grad_out / n_valid. held_h: grad_hidden, or None; kind: 0 bf16, 1 bf16
// whose gradient is fp32, 2 fp32. Returns (grad_hidden, grad_weight).
py::tuple ce_backward(const at::Tensor& grad_out, const at::Tensor& out2, const c10::optional<at::Tensor>& held_h,
                      int kind, const c10::optional<at::Tensor>& grad_w, const std::vector<at::Tensor>& chunks,
                      bool accumulated, uintptr_t stream_handle) {
  HANDLE_TH_ERRORS
  const Abi& a = abi();
  at::Tensor gw = grad_w ? *grad_w : at::Tensor(), gh = held_h ? *held_h : at::Tensor();
  without_gil([&] {
    at::Tensor g = grad_out.detach().to(at::kFloat).contiguous();
    const auto f32 = out2.options();
    if (!gw.defined() && !chunks.empty()) gw = at::empty(chunks[0].sizes(), f32);
    if (kind == 1 && gh.defined()) gh = at::empty(gh.sizes(), f32);
    std::vector<const void*> p;
    for (const at::Tensor& t : chunks) p.push_back(ptr(t));
    check(a.finish(ptr(gw), p.data(), static_cast<int>(p.size()), gw.defined() ? gw.numel() : 0, accumulated,
                   held_h ? ptr(*held_h) : nullptr, ptr(gh), gh.defined() ? gh.numel() : 0, kind, ptr(g),
                   out2.data_ptr<float>() + 1, reinterpret_cast<void*>(stream_handle)),
          "tm_ce_finish");
  });
  return py::make_tuple(or_none(gh), or_none(gw));
  END_HANDLE_TH_ERRORS_PYBIND
}

}  // namespace

void tm_ce_host_bind(py::module_& m) {
  m.def("ce_bind", &ce_bind, "addresses of the C ABI's fused CE entry points, and the exception class of a failed call");
  m.def("ce_forward", &ce_forward, "the chunks of one fused linear + CE call");
  m.def("ce_backward", &ce_backward, "backward of one fused linear + CE call");
}

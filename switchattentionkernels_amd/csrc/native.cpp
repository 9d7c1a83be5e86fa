// The host path of the package's hot calls: allocate the results, launch
// through the C ABI, wait for the one value that a call needs on the host.
// Bound with pybind11 for the Python layer, which keeps the API, its argument
// checks and their messages; nothing here is reached with arguments that layer
// has not accepted.
//
// Bound by call overhead: with ctypes and Python bookkeeping a forward took
// about 20 us of host time between the routing's read-back and its launch, in
// which the GPU is idle; these take about 8.

#include <ATen/core/CachingHostAllocator.h>
#include <torch/extension.h>

#include <string>
#include <tuple>
#include <vector>

#include "swattn.h"
#include "swattn_internal.h"

namespace {

using at::Tensor;
using std::optional;
namespace py = pybind11;

void check(int status, const char* what) {
  TORCH_CHECK(status == SWATTN_OK, what, " failed with status ", status, ": ", swattn_last_error());
}

void* as_stream(int64_t s) { return reinterpret_cast<void*>(static_cast<intptr_t>(s)); }

Tensor bytes(const Tensor& like, size_t n) {
  return at::empty({static_cast<int64_t>(n)}, like.options().dtype(at::kByte));
}

// An output like t: the one that the Python layer made, where a tensor subclass
// has a say in that, or a new one.
Tensor like(const Tensor& t, const optional<Tensor>& made) {
  return made.has_value() ? *made : at::empty(t.sizes(), t.options());
}

const int32_t* i32(const Tensor& t) { return static_cast<const int32_t*>(t.const_data_ptr()); }
const int32_t* i32(const optional<Tensor>& t) { return t.has_value() ? i32(*t) : nullptr; }

// Pinned host memory for a compaction's counts.  One buffer per thread: a call
// waits for its counts before it returns, so that a thread has at most one
// compaction in flight.  After a HIP error a kernel may still be queued that
// reports there: the buffer is then left to it for good.
thread_local c10::DataPtr t_words;
int32_t* host_words() {
  if (!t_words)
    t_words = at::getHostAllocator(at::kCUDA)->allocate(SWATTN_COMPACT_HOST_WORDS * sizeof(int32_t));
  return static_cast<int32_t*>(t_words.get());
}
void abandon_host_words() {
  (void)t_words.release_context();
  t_words = c10::DataPtr();
}

// (full, local) of a byte mask (dtype -1) or of router logits.
std::tuple<Tensor, Tensor> compact(const Tensor& x, int64_t dtype, double threshold,
                                   int64_t stream) {
  const int64_t n = x.numel();
  const Tensor out = at::empty({n}, x.options().dtype(at::kInt));
  const size_t ws_bytes = swattn_compact_workspace_bytes(n);
  Tensor ws;
  if (ws_bytes > 0) ws = bytes(x, ws_bytes);
  int32_t* host = host_words();
  int status = 0;
  {
    pybind11::gil_scoped_release release;
    status = swattn_compact_wait(x.const_data_ptr(), static_cast<int32_t>(dtype), n,
                                 static_cast<float>(threshold), out.data_ptr<int32_t>(), host,
                                 ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes,
                                 as_stream(stream));
  }
  if (status > 0) abandon_host_words();
  check(status, dtype < 0 ? "swattn_compact" : "swattn_compact_logits");
  const int64_t nf = host[0];
  return {out.narrow(0, 0, nf), out.narrow(0, nf, n - nf)};
}

// Whether q, k, v meet every precondition of the prefill (the Python layer
// finds out which one fails and raises for it, also for arguments that are no
// tensors).
bool qkv_ok(const py::object& qo, const py::object& ko, const py::object& vo) {
  if (!THPVariable_Check(qo.ptr()) || !THPVariable_Check(ko.ptr()) || !THPVariable_Check(vo.ptr()))
    return false;
  const Tensor& q = THPVariable_Unpack(qo.ptr());
  const Tensor& k = THPVariable_Unpack(ko.ptr());
  const Tensor& v = THPVariable_Unpack(vo.ptr());
  return q.scalar_type() == at::kBFloat16 && k.scalar_type() == at::kBFloat16 &&
         v.scalar_type() == at::kBFloat16 && q.is_cuda() && k.is_cuda() && v.is_cuda() &&
         q.layout() == at::kStrided && k.layout() == at::kStrided && v.layout() == at::kStrided &&
         q.is_contiguous() && k.is_contiguous() && v.is_contiguous() && q.dim() == 4 &&
         k.dim() == 4 && v.dim() == 4 && k.sizes() == v.sizes() && q.size(0) == k.size(0) &&
         q.size(3) == 128 && k.size(3) == 128 && k.size(2) > 0 && q.size(2) % k.size(2) == 0 &&
         q.device() == k.device() && q.device() == v.device();
}

std::tuple<Tensor, Tensor> prefill_forward(const Tensor& q, const Tensor& k, const Tensor& v,
                                           const Tensor& full, const Tensor& local,
                                           const optional<Tensor>& full_starts,
                                           const optional<Tensor>& local_starts,
                                           const optional<Tensor>& causal_ends, int64_t window,
                                           double scale_log2, int64_t stream,
                                           const optional<Tensor>& out_made) {
  const int32_t batch = static_cast<int32_t>(q.size(0)), hq = static_cast<int32_t>(q.size(2));
  const int32_t hkv = static_cast<int32_t>(k.size(2)), dim = static_cast<int32_t>(q.size(3));
  const int64_t sq = q.size(1), skv = k.size(1), nf = full.numel(), nl = local.numel();
  const Tensor out = like(q, out_made);
  const Tensor lse = at::empty({q.size(0), sq, q.size(2)}, q.options().dtype(at::kFloat));
  const int32_t w = static_cast<int32_t>(window);
  // The larger workspace that lets the kernel split long full items by key
  // range when they would otherwise set its length (few KV heads).
  const size_t ws_bytes =
      swattn_prefill_split_workspace_bytes(batch, sq, skv, hq, hkv, dim, w, nf, nl);
  const Tensor ws = bytes(q, ws_bytes);
  int status = 0;
  {
    pybind11::gil_scoped_release release;
    status = swattn_prefill_fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), i32(full),
                   nf, i32(local), nl, i32(full_starts), i32(local_starts),
                   i32(causal_ends), out.data_ptr(), lse.data_ptr<float>(), batch, sq, skv,
                   hq, hkv, dim, w, static_cast<float>(scale_log2), ws.data_ptr(), ws_bytes,
                   as_stream(stream));
  }
  check(status, "swattn_prefill_fwd");
  return {out, lse};
}

// The seven fields of a SwitchAttentionMetadata, in its order; the sequences'
// offsets, checked and at most SWATTN_METADATA_HOST_MAX_SEQS of them, travel as
// kernel arguments.
std::vector<Tensor> metadata(const std::vector<int32_t>& cu_q, const std::vector<int32_t>& cu_kv,
                             int64_t q_len, int64_t kv_len, int64_t window, at::Device device,
                             int64_t stream) {
  const auto opts = at::TensorOptions().dtype(at::kInt).device(device);
  std::vector<Tensor> f;
  f.reserve(7);
  for (const int64_t n : {q_len, kv_len, q_len, kv_len, q_len, q_len, q_len})
    f.push_back(at::empty({n}, opts));
  auto out = [&](int i) { return f[i].data_ptr<int32_t>(); };
  check(swattn_build_metadata_host(cu_q.data(), cu_kv.data(), static_cast<int32_t>(cu_q.size()) - 1,
                                   q_len, kv_len, static_cast<int32_t>(window), out(0), out(1),
                                   out(2), out(3), out(4), out(5), out(6), as_stream(stream)),
        "swattn_build_metadata");
  return f;
}

std::tuple<Tensor, Tensor, Tensor> prefill_backward(
    const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse,
    const Tensor& grad, const Tensor& full, const Tensor& local,
    const optional<Tensor>& full_starts, const optional<Tensor>& local_starts,
    const optional<Tensor>& causal_ends, int64_t window, double scale_log2, int64_t stream,
    const optional<Tensor>& dq_made, const optional<Tensor>& dk_made,
    const optional<Tensor>& dv_made) {
  const int32_t batch = static_cast<int32_t>(q.size(0)), hq = static_cast<int32_t>(q.size(2));
  const int32_t hkv = static_cast<int32_t>(k.size(2)), dim = static_cast<int32_t>(q.size(3));
  const int64_t sq = q.size(1), skv = k.size(1), nf = full.numel(), nl = local.numel();
  // The lists cover every query position once (checked by the caller), and the
  // kernels write every listed row (0 for a row with no key): no fill.
  const Tensor dq = like(q, dq_made), dk = like(k, dk_made), dv = like(v, dv_made);
  const int32_t w = static_cast<int32_t>(window);
  const size_t ws_bytes = swattn_prefill_bwd_workspace_bytes(batch, skv, hq, hkv, dim, w, nf, nl);
  const Tensor ws = bytes(q, ws_bytes > 0 ? ws_bytes : 1);
  int status = 0;
  {
    pybind11::gil_scoped_release release;
    status = swattn_prefill_bwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                   out.const_data_ptr(), lse.const_data_ptr<float>(),
                   grad.const_data_ptr(), i32(full), nf, i32(local), nl, i32(full_starts),
                   i32(local_starts), i32(causal_ends), dq.data_ptr(), dk.data_ptr(),
                   dv.data_ptr(), batch, sq, skv, hq, hkv, dim, w,
                   static_cast<float>(scale_log2), ws.data_ptr(), ws_bytes,
                   as_stream(stream));
  }
  check(status, "swattn_prefill_bwd");
  return {dq, dk, dv};
}

std::tuple<Tensor, Tensor> decode_forward(const Tensor& q, const Tensor& k, const Tensor& v,
                                          const Tensor& lens, const Tensor& full, int64_t window,
                                          double scale_log2, int64_t stream,
                                          const optional<Tensor>& out_made) {
  const int32_t batch = static_cast<int32_t>(q.size(0)), hq = static_cast<int32_t>(q.size(2));
  const int32_t hkv = static_cast<int32_t>(k.size(2)), dim = static_cast<int32_t>(q.size(3));
  const Tensor out = like(q, out_made);
  const Tensor lse = at::empty({q.size(0), 1, q.size(2)}, q.options().dtype(at::kFloat));
  const size_t ws_bytes = swattn_decode_workspace_bytes(batch, k.size(1), hq, hkv);
  const Tensor ws = bytes(q, ws_bytes);
  int status = 0;
  {
    pybind11::gil_scoped_release release;
    status = swattn_decode_fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), i32(lens),
                  static_cast<const uint8_t*>(full.const_data_ptr()), out.data_ptr(),
                  lse.data_ptr<float>(), batch, k.size(1), hq, hkv, dim,
                  static_cast<int32_t>(window), static_cast<float>(scale_log2),
                  ws.data_ptr(), ws_bytes, as_stream(stream));
  }
  check(status, "swattn_decode_fwd");
  return {out, lse};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("compact", &compact);
  m.def("qkv_ok", &qkv_ok);
  m.def("prefill_forward", &prefill_forward);
  m.def("metadata", &metadata);
  m.def("prefill_backward", &prefill_backward);
  m.def("decode_forward", &decode_forward);
}

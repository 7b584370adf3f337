// gqa_host.cpp — torch-tensor bindings of the split-KV decode call and of
// the paged-cache launches.
//
// The decode route of gqa_flash_attn (reference gqa_kernels/dispatch.py:49-56,
// gqa_split.py:153-194) is one gqa_split_launch per step.  Driven through
// ctypes, building its 21 arguments (four stride arrays, pointers read off
// the tensors one Python call at a time) costs more host time per step than
// the GPU spends on a short cache (8192 keys: ~12.5 us of host time against
// ~9.8 us of kernels), so a loop of decode steps waits on the host.  This
// binding takes the tensors themselves, reads pointers, strides and the
// current HIP stream natively, allocates the output (and LSE) with torch,
// and calls the same C entry point (include/gqa_attn.h) — the library
// boundary is unchanged; only the marshalling moves out of Python.  The
// paged routes (paged_forward: split-KV first pass + combine, single pass,
// key chunks) and the paged cache write get the same treatment: through
// ctypes a paged decode step spent ~18 us on the host against ~10 us of
// kernels.
//
// Host-only C++ (no kernels); built by build.py into gqa_kernels/ next to
// libgqa_hip.so, which it links against.
#include <torch/extension.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/python_arg_parser.h>

#include <algorithm>
#include <array>
#include <stdexcept>
#include <string>
#include <unordered_map>

#include "gqa_attn.h"

namespace {

void strides_of(const at::Tensor& t, int64_t (&s)[4]) {
  for (int i = 0; i < 4; ++i) s[i] = t.stride(i);
}

// q, k, v: 4-d (B, H, S, D) tensors the kernels can read (unit last-dim
// stride, 16-byte aligned rows — the caller's fast-path test, checked again
// by the C entry point); ws: the stream's fp32 workspace of at least
// gqa_split_workspace_bytes(...) bytes.  Returns o, or (o, lse).
py::object split_decode(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& ws,
                        int64_t splits, bool causal, double scale_log2, int64_t dtype, bool return_lse) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) throw std::invalid_argument("split_decode: 4-d q, k, v expected");
  if (ws.scalar_type() != at::kFloat) throw std::invalid_argument("split_decode: fp32 workspace expected");
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), D = q.size(3);
  const int64_t Hkv = k.size(1), Skv = k.size(2);
  at::Tensor o = at::empty_like(q);
  at::Tensor lse;
  if (return_lse) lse = at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat));
  int64_t qs[4], ks[4], vs[4], os[4];
  strides_of(q, qs);
  strides_of(k, ks);
  strides_of(v, vs);
  strides_of(o, os);
  hipStream_t stream = c10::hip::getCurrentHIPStream(q.get_device()).stream();
  const int rc = gqa_split_launch(q.data_ptr(), qs, k.data_ptr(), ks, v.data_ptr(), vs, o.data_ptr(), os,
                                  return_lse ? lse.data_ptr<float>() : nullptr, ws.data_ptr<float>(),
                                  static_cast<int>(splits), static_cast<int>(B), static_cast<int>(Hq),
                                  static_cast<int>(Hkv), static_cast<int>(Sq), static_cast<int>(Skv),
                                  static_cast<int>(D), static_cast<float>(scale_log2), causal ? 1 : 0,
                                  static_cast<int>(dtype), stream);
  if (rc != GQA_OK) {
    // The package's own error path (gqa_kernels._lib.check raises GQAError
    // with the library's message), as for the ctypes-bound entry points.
    py::module_::import("gqa_kernels._lib").attr("check")(rc);
    throw std::runtime_error(std::string("gqa_split_launch failed: ") + gqa_strerror(rc));
  }
  if (return_lse) return py::make_tuple(o, lse);
  return py::cast(o);
}

// gqa_split_flat_launch into a fresh o (and lse): ws of at least
// gqa_split_flat_workspace_bytes(...) bytes.  None when the call is not one the
// flat split takes (GQA_E_FLAT).
py::object split_flat(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& ws,
                      int64_t slots, bool causal, double scale_log2, int64_t dtype, bool return_lse) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) throw std::invalid_argument("split_flat: 4-d q, k, v expected");
  if (ws.scalar_type() != at::kFloat) throw std::invalid_argument("split_flat: fp32 workspace expected");
  at::Tensor o = at::empty_like(q);
  at::Tensor lse;
  if (return_lse) lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
  int64_t qs[4], ks[4], vs[4], os[4];
  strides_of(q, qs);
  strides_of(k, ks);
  strides_of(v, vs);
  strides_of(o, os);
  hipStream_t stream = c10::hip::getCurrentHIPStream(q.get_device()).stream();
  const int rc = gqa_split_flat_launch(
      q.data_ptr(), qs, k.data_ptr(), ks, v.data_ptr(), vs, o.data_ptr(), os,
      return_lse ? lse.data_ptr<float>() : nullptr, ws.data_ptr<float>(), static_cast<int>(slots),
      static_cast<int>(q.size(0)), static_cast<int>(q.size(1)), static_cast<int>(k.size(1)),
      static_cast<int>(q.size(2)), static_cast<int>(k.size(2)), static_cast<int>(q.size(3)),
      static_cast<float>(scale_log2), causal ? 1 : 0, static_cast<int>(dtype), stream);
  if (rc == GQA_E_FLAT) return py::none();
  if (rc != GQA_OK) {
    py::module_::import("gqa_kernels._lib").attr("check")(rc);
    throw std::runtime_error(std::string("gqa_split_flat_launch failed: ") + gqa_strerror(rc));
  }
  if (return_lse) return py::make_tuple(o, lse);
  return py::cast(o);
}

[[noreturn]] void raise_rc(int rc, const char* what) {
  py::module_::import("gqa_kernels._lib").attr("check")(rc);
  throw std::runtime_error(std::string(what) + " failed: " + gqa_strerror(rc));
}

// The kernel routes of paged attention (gqa_kernels.paged.paged_attention,
// after its checks and route choice), launched from the tensors:
//   route 0: gqa_paged_split_first_launch into ws, then the combine into out
//            (gqa_split_reduce_varlen_launch with variable query lengths,
//            else gqa_split_reduce_lse_launch or gqa_split_reduce_launch);
//   route 1: gqa_paged_fwd_launch, or with `splits` > 0 split query blocks
//            gqa_paged_fwd_split_launch (ws, zeroed counters);
//   route 2: gqa_paged_fwd_chunks_launch (ws, `splits` key chunks);
//   route 3: gqa_paged_split_flat_launch (ws, `splits` slots);
//   route 4: gqa_paged_fwd_short_launch.
// Returns false (nothing launched) when route 3 does not take the call.
// q and out are (batch, heads, seq_q, head_dim), or token-major
// (tokens, heads, head_dim) when q_start / q_len are given.
bool paged_forward(int64_t route, const at::Tensor& q, const at::Tensor& k_cache, const at::Tensor& v_cache,
                   const at::Tensor& block_table, int64_t table_stride, const at::Tensor& seq_lens,
                   const std::optional<at::Tensor>& q_start, const std::optional<at::Tensor>& q_len,
                   int64_t max_seq_len, const at::Tensor& out, const std::optional<at::Tensor>& lse,
                   const std::optional<at::Tensor>& ws, const std::optional<at::Tensor>& counters,
                   int64_t splits, int64_t batch, int64_t seq_q,
                   double scale_log2, bool causal, int64_t dtype) {
  if (k_cache.dim() != 4 || v_cache.dim() != 4) throw std::invalid_argument("paged_forward: 4-d caches expected");
  const bool varlen = q_start.has_value() && q_len.has_value();
  if (varlen ? q.dim() != 3 || out.dim() != 3 : q.dim() != 4 || out.dim() != 4)
    throw std::invalid_argument("paged_forward: q / out rank does not match the query layout");
  if (route != 4 && (route != 1 || splits > 0) && !ws.has_value()) throw std::invalid_argument("paged_forward: workspace expected");
  if (route == 1 && splits > 0 && !counters.has_value())
    throw std::invalid_argument("paged_forward: counters expected");
  const int H = static_cast<int>(q.size(1)), D = static_cast<int>(q.size(-1));
  const int Hkv = static_cast<int>(k_cache.size(2)), bs = static_cast<int>(k_cache.size(1));
  int64_t qs[4], os[4], ks[4], vs[4];
  if (varlen) {
    const int64_t qv[4] = {0, q.stride(1), q.stride(0), 1}, ov[4] = {0, out.stride(1), out.stride(0), 1};
    for (int i = 0; i < 4; ++i) qs[i] = qv[i], os[i] = ov[i];
  } else {
    strides_of(q, qs);
    strides_of(out, os);
  }
  strides_of(k_cache, ks);
  strides_of(v_cache, vs);
  const int* qst = varlen ? q_start->data_ptr<int>() : nullptr;
  const int* qln = varlen ? q_len->data_ptr<int>() : nullptr;
  float* lse_p = lse.has_value() ? lse->data_ptr<float>() : nullptr;
  float* ws_p = ws.has_value() ? ws->data_ptr<float>() : nullptr;
  const int B = static_cast<int>(batch), Sq = static_cast<int>(seq_q), S = static_cast<int>(splits);
  const int dt = static_cast<int>(dtype), ms = static_cast<int>(max_seq_len), ts = static_cast<int>(table_stride);
  const float sl2 = static_cast<float>(scale_log2);
  hipStream_t stream = c10::hip::getCurrentHIPStream(q.get_device()).stream();
  const int* table = block_table.data_ptr<int>();
  const int* lens = seq_lens.data_ptr<int>();
  int rc;
  if (route == 1 && S > 0) {
    rc = gqa_paged_fwd_split_launch(q.data_ptr(), qs, k_cache.data_ptr(), ks, v_cache.data_ptr(), vs, table, ts,
                                    lens, qst, qln, bs, ms, out.data_ptr(), os, lse_p, ws_p,
                                    counters->data_ptr<int>(), S, B, H, Hkv, Sq, D, sl2, causal ? 1 : 0, dt, stream);
    if (rc != GQA_OK) raise_rc(rc, "gqa_paged_fwd_split_launch");
    return true;
  }
  if (route == 1) {
    rc = gqa_paged_fwd_launch(q.data_ptr(), qs, k_cache.data_ptr(), ks, v_cache.data_ptr(), vs, table, ts, lens,
                              qst, qln, bs, ms, out.data_ptr(), os, lse_p, B, H, Hkv, Sq, D, sl2, causal ? 1 : 0,
                              dt, stream);
    if (rc != GQA_OK) raise_rc(rc, "gqa_paged_fwd_launch");
    return true;
  }
  if (route == 2) {
    rc = gqa_paged_fwd_chunks_launch(q.data_ptr(), qs, k_cache.data_ptr(), ks, v_cache.data_ptr(), vs, table, ts,
                                     lens, qst, qln, bs, ms, out.data_ptr(), os, lse_p, ws_p, S, B, H, Hkv, Sq, D,
                                     sl2, causal ? 1 : 0, dt, stream);
    if (rc != GQA_OK) raise_rc(rc, "gqa_paged_fwd_chunks_launch");
    return true;
  }
  if (route == 3) {
    rc = gqa_paged_split_flat_launch(q.data_ptr(), qs, k_cache.data_ptr(), ks, v_cache.data_ptr(), vs, table, ts,
                                     lens, qst, qln, bs, ms, out.data_ptr(), os, lse_p, ws_p, S, B, H, Hkv, Sq, D,
                                     sl2, causal ? 1 : 0, dt, stream);
    if (rc == GQA_E_FLAT) return false;
    if (rc != GQA_OK) raise_rc(rc, "gqa_paged_split_flat_launch");
    return true;
  }
  if (route == 4) {
    rc = gqa_paged_fwd_short_launch(q.data_ptr(), qs, k_cache.data_ptr(), ks, v_cache.data_ptr(), vs, table, ts, lens,
                                    qst, qln, bs, ms, out.data_ptr(), os, lse_p, B, H, Hkv, Sq, D, sl2,
                                    causal ? 1 : 0, dt, stream);
    if (rc != GQA_OK) raise_rc(rc, "gqa_paged_fwd_short_launch");
    return true;
  }
  if (route != 0) throw std::invalid_argument("paged_forward: route must be 0 to 4");
  rc = gqa_paged_split_first_launch(q.data_ptr(), qs, k_cache.data_ptr(), ks, v_cache.data_ptr(), vs, table, ts,
                                    lens, qst, qln, bs, ms, ws_p, S, B, H, Hkv, Sq, D, sl2, causal ? 1 : 0, dt,
                                    stream);
  if (rc != GQA_OK) raise_rc(rc, "gqa_paged_split_first_launch");
  if (varlen)
    rc = gqa_split_reduce_varlen_launch(ws_p, S, out.data_ptr(), os, lse_p, qst, qln, B, H, Sq, D, dt, stream);
  else if (lse_p != nullptr)
    rc = gqa_split_reduce_lse_launch(ws_p, S, out.data_ptr(), os, lse_p, B, H, Sq, D, dt, stream);
  else
    rc = gqa_split_reduce_launch(ws_p, S, out.data_ptr(), os, B, H, Sq, D, dt, stream);
  if (rc != GQA_OK) raise_rc(rc, "gqa_split_reduce_launch");
  return true;
}

// gqa_paged_cache_write_launch from the tensors (gqa_kernels.paged.write_kv
// after its checks): key / value (tokens, kv heads, head_dim), int64 slots.
void cache_write(const at::Tensor& key, const at::Tensor& value, const at::Tensor& k_cache,
                 const at::Tensor& v_cache, const at::Tensor& slot_mapping, int64_t dtype) {
  if (key.dim() != 3 || value.dim() != 3 || k_cache.dim() != 4 || v_cache.dim() != 4)
    throw std::invalid_argument("cache_write: 3-d key / value and 4-d caches expected");
  const int64_t kst[3] = {key.stride(0), key.stride(1), key.stride(2)};
  const int64_t vst[3] = {value.stride(0), value.stride(1), value.stride(2)};
  int64_t kcs[4], vcs[4];
  strides_of(k_cache, kcs);
  strides_of(v_cache, vcs);
  hipStream_t stream = c10::hip::getCurrentHIPStream(key.get_device()).stream();
  const int rc = gqa_paged_cache_write_launch(
      key.data_ptr(), kst, value.data_ptr(), vst, k_cache.data_ptr(), kcs, v_cache.data_ptr(), vcs,
      slot_mapping.data_ptr<int64_t>(), static_cast<int>(key.size(0)), static_cast<int>(key.size(1)),
      static_cast<int>(key.size(2)), static_cast<int>(k_cache.size(1)), static_cast<int>(dtype), stream);
  if (rc != GQA_OK) raise_rc(rc, "gqa_paged_cache_write_launch");
}

// ---------------------------------------------------------------------------
// Whole calls.  gqa_flash_attn and paged_attention spend 10-20 us per call in
// Python on checks, the route and the launch arguments, more than the kernels
// of a short call take on the GPU (333 tokens: 16 us of host time beside 9.9
// us).  These entries do the usual case natively: every check passes, the
// route of these shapes is known (set_plan, from Python's rules) and the
// stream's buffers are large enough.  Anything else returns None with
// nothing launched, and Python takes the call: it raises, copies, chooses the
// route (and registers it here) or grows the buffer.
// ---------------------------------------------------------------------------
enum Kind : int { kSplit = 0, kSingle = 1, kChunks = 2, kFlat = 3, kShort = 4 };

struct Plan {
  int kind, n;         // n: splits, split blocks, key chunks or slots
  float scale_log2;    // gqa_flash_attn: head_dim^-0.5 * log2(e)
};

using Key = std::array<int64_t, 12>;
struct KeyHash {
  size_t operator()(const Key& k) const {
    uint64_t h = 1469598103934665603ull;
    for (int64_t v : k) h = (h ^ (uint64_t)v) * 1099511628211ull;
    return (size_t)(h ^ (h >> 32));
  }
};
// Guarded by the GIL, which every use of the table holds; bounded as Python's
// own route caches are.
std::unordered_map<Key, Plan, KeyHash> g_plans;

void set_plan(const std::vector<int64_t>& key, int64_t kind, int64_t n, double scale_log2) {
  Key k{};
  if (key.size() != k.size()) throw std::invalid_argument("set_plan: key length");
  std::copy(key.begin(), key.end(), k.begin());
  if (g_plans.size() >= 8192) g_plans.clear();
  g_plans[k] = Plan{static_cast<int>(kind), static_cast<int>(n), static_cast<float>(scale_log2)};
}

// A plain tensor (no subclass, wrapper or active mode that would have to see
// the call), or nullptr.
const at::Tensor* plain(const py::handle& h) {
  if (!THPVariable_CheckExact(h.ptr())) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(h.ptr());
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || at::isTensorSubclassLike(t)) return nullptr;
  return &t;
}
bool modes_active() {
  return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set();
}
bool half_type(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
int dtype_code(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 ? GQA_DTYPE_BF16 : GQA_DTYPE_FP16; }

// Unit last stride, every other stride and the pointer multiples of 16 bytes
// (2-byte elements).
bool rows_ready(const at::Tensor& t) {
  const int64_t d = t.dim();
  if (t.stride(d - 1) != 1) return false;
  uint64_t bits = reinterpret_cast<uintptr_t>(t.data_ptr());
  for (int64_t i = 0; i < d - 1; ++i) bits |= 2 * static_cast<uint64_t>(t.stride(i));
  return (bits & 15) == 0;
}

// The stream's buffer of at least `bytes` bytes from gqa_split's dictionary,
// or nullptr.
void* stream_buffer(const py::dict& buffers, int64_t dev, hipStream_t stream, size_t bytes) {
  const py::tuple key = py::make_tuple(dev, reinterpret_cast<intptr_t>(stream));
  PyObject* v = PyDict_GetItemWithError(buffers.ptr(), key.ptr());
  if (v == nullptr) {
    PyErr_Clear();
    return nullptr;
  }
  if (!THPVariable_Check(v)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(v);
  return t.nbytes() >= bytes ? t.data_ptr() : nullptr;
}

bool capturing() {
  return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

void check_rc(int rc, const char* what) {
  if (rc != GQA_OK) raise_rc(rc, what);
}

// gqa_flash_attn(q, k, v, causal, return_lse), or None.  workspaces, counters:
// gqa_split's per-stream buffers.
py::object flash_attn(const py::handle& hq, const py::handle& hk, const py::handle& hv, bool causal, bool return_lse,
                      const py::dict& workspaces, const py::dict& counters) {
  const at::Tensor *pq = plain(hq), *pk = plain(hk), *pv = plain(hv);
  if (pq == nullptr || pk == nullptr || pv == nullptr || modes_active()) return py::none();
  const at::Tensor &q = *pq, &k = *pk, &v = *pv;
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || !half_type(q) || k.scalar_type() != q.scalar_type() ||
      v.scalar_type() != q.scalar_type() || v.sizes() != k.sizes())
    return py::none();
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), D = q.size(3), Hkv = k.size(1), Skv = k.size(2);
  const int64_t dev = q.get_device();
  if (k.size(0) != B || k.size(3) != D || k.get_device() != dev || v.get_device() != dev ||
      c10::hip::current_device() != dev)
    return py::none();
  const auto found = g_plans.find(Key{0, B, Hq, Hkv, Sq, Skv, D, causal, dev});
  if (found == g_plans.end() || !rows_ready(q) || !rows_ready(k) || !rows_ready(v)) return py::none();
  const Plan p = found->second;
  if (p.kind != kSingle && (Skv + 192) * std::max(k.stride(2), v.stride(2)) >= ((int64_t)1 << 30)) return py::none();
  hipStream_t stream = c10::hip::getCurrentHIPStream(dev).stream();

  void *ws = nullptr, *cnt = nullptr;
  size_t need = 0;
  if (p.kind == kSplit || p.kind == kChunks)
    need = gqa_split_workspace_bytes(B, Hq, Sq, D, p.n);
  else if (p.kind == kFlat)
    need = gqa_split_flat_workspace_bytes(B, Hq, Sq, D, p.n);
  else if (p.kind == kSingle)
    need = gqa_fwd_split_workspace_bytes(B, Hkv, D, p.n);
  // (A captured call gets partials and counters of its own, in Python.)
  if (need > 0 && (capturing() || (ws = stream_buffer(workspaces, dev, stream, need)) == nullptr)) return py::none();
  if (p.kind == kSingle || p.kind == kChunks) {
    const size_t n = gqa_fwd_split_counters_count(B, Hkv, p.kind == kSingle ? p.n : 0);
    if (capturing() || (cnt = stream_buffer(counters, dev, stream, n * sizeof(int))) == nullptr) return py::none();
  }
  at::Tensor o = at::empty_like(q);
  if (!rows_ready(o)) return py::none();
  at::Tensor lse;
  if (return_lse) lse = at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat));
  float* lse_p = return_lse ? lse.data_ptr<float>() : nullptr;
  int64_t qs[4], ks[4], vs[4], os[4];
  strides_of(q, qs);
  strides_of(k, ks);
  strides_of(v, vs);
  strides_of(o, os);
  const int b = B, hq_ = Hq, hkv = Hkv, sq = Sq, skv = Skv, d = D, c = causal ? 1 : 0, dt = dtype_code(q);
  const float sl2 = p.scale_log2;
  float* wsf = static_cast<float*>(ws);
  int* cnti = static_cast<int*>(cnt);
  const void *qp = q.data_ptr(), *kp = k.data_ptr(), *vp = v.data_ptr();
  void* op = o.data_ptr();
  int rc;
  const char* what;
  if (p.kind == kSplit) {
    what = "gqa_split_launch";
    rc = gqa_split_launch(qp, qs, kp, ks, vp, vs, op, os, lse_p, wsf, p.n, b, hq_, hkv, sq, skv, d, sl2, c, dt, stream);
  } else if (p.kind == kFlat) {
    what = "gqa_split_flat_launch";
    rc = gqa_split_flat_launch(qp, qs, kp, ks, vp, vs, op, os, lse_p, wsf, p.n, b, hq_, hkv, sq, skv, d, sl2, c, dt,
                               stream);
    if (rc == GQA_E_FLAT) return py::none();
  } else if (p.kind == kChunks) {
    what = "gqa_fwd_chunks_launch";
    rc = gqa_fwd_chunks_launch(qp, qs, kp, ks, vp, vs, op, os, lse_p, wsf, cnti, p.n, b, hq_, hkv, sq, skv, d, sl2, c,
                               dt, stream);
  } else {
    // One launch: other threads run while it waits for room in a full queue.
    // (The two launches of the calls above share the stream's workspace, which
    // a call of another thread must not enter in between.)
    py::gil_scoped_release others;
    what = p.kind == kShort ? "gqa_fwd_short_launch" : "gqa_fwd_split_launch";
    rc = p.kind == kShort
             ? gqa_fwd_short_launch(qp, qs, kp, ks, vp, vs, op, os, lse_p, b, hq_, hkv, sq, skv, d, sl2, c, dt, stream)
             : gqa_fwd_split_launch(qp, qs, kp, ks, vp, vs, op, os, lse_p, wsf, cnti, p.n, b, hq_, hkv, sq, skv, d, sl2,
                                    c, dt, stream);
  }
  check_rc(rc, what);
  if (return_lse) return py::make_tuple(o, lse);
  return py::cast(o);
}

// (num_blocks, block_size, Hkv, D) caches paged_attention and write_kv accept.
bool caches_ready(const at::Tensor& kc, const at::Tensor& vc) {
  if (kc.dim() != 4 || vc.dim() != 4 || kc.sizes() != vc.sizes() || kc.scalar_type() != vc.scalar_type() ||
      kc.get_device() != vc.get_device() || !half_type(kc))
    return false;
  const int64_t bs = kc.size(1);
  return bs >= 1 && bs <= GQA_MAX_BLOCK_SIZE && (bs & (bs - 1)) == 0 && rows_ready(kc) && rows_ready(vc);
}
bool int_rows(const at::Tensor* t, int64_t n, int64_t dev) {
  return t != nullptr && t->scalar_type() == at::kInt && t->dim() == 1 && t->size(0) == n && t->is_contiguous() &&
         t->get_device() == dev;
}

// paged_attention on its default route, or None.  max_seq_len and
// max_query_len < 0: not given; qstart None: uniform query lengths.
py::object paged_attn(const py::handle& hq, const py::handle& hkc, const py::handle& hvc, const py::handle& htab,
                      const py::handle& hlens, bool causal, int64_t max_seq_len, double scale_log2, bool return_lse,
                      const py::handle& hout, const py::handle& hqs, const py::handle& hql, int64_t max_query_len,
                      const py::dict& workspaces, const py::dict& counters) {
  const at::Tensor *pq = plain(hq), *pkc = plain(hkc), *pvc = plain(hvc), *ptab = plain(htab), *plens = plain(hlens);
  if (pq == nullptr || pkc == nullptr || pvc == nullptr || ptab == nullptr || plens == nullptr || modes_active())
    return py::none();
  const at::Tensor &q = *pq, &kc = *pkc, &vc = *pvc, &tab = *ptab, &lens = *plens;
  const bool varlen = !hqs.is_none();
  if (q.dim() != (varlen ? 3 : 4) || !caches_ready(kc, vc) || q.scalar_type() != kc.scalar_type() || !rows_ready(q))
    return py::none();
  const int64_t dev = q.get_device(), H = q.size(1), D = q.size(-1), Hkv = kc.size(2), bs = kc.size(1);
  const int64_t B = varlen ? (lens.dim() == 1 ? lens.size(0) : -1) : q.size(0);
  const int64_t Sq = varlen ? max_query_len : q.size(2);
  const at::Tensor *qst = nullptr, *qln = nullptr;
  if (varlen) {
    qst = plain(hqs);
    qln = plain(hql);
    if (Sq < 0 || !int_rows(qst, B, dev) || !int_rows(qln, B, dev)) return py::none();
  }
  if (kc.get_device() != dev || kc.size(3) != D || !int_rows(&lens, B, dev) || tab.scalar_type() != at::kInt ||
      tab.dim() != 2 || tab.size(0) != B || tab.get_device() != dev || tab.stride(1) != 1 ||
      (B > 1 && tab.stride(0) < tab.size(1)) || c10::hip::current_device() != dev)
    return py::none();
  const int64_t capacity = tab.size(1) * bs;
  if (max_seq_len < 0) max_seq_len = capacity;
  if (max_seq_len > capacity) return py::none();
  const bool interleaved = kc.stride(1) != D || vc.stride(1) != D;
  const auto found = g_plans.find(Key{1, B, H, Hkv, Sq, max_seq_len, D, causal, dev, bs, interleaved, varlen});
  if (found == g_plans.end()) return py::none();
  const Plan p = found->second;
  if (p.kind == kShort && std::max(kc.stride(1), vc.stride(1)) >= ((int64_t)1 << 24)) return py::none();
  hipStream_t stream = c10::hip::getCurrentHIPStream(dev).stream();
  void *ws = nullptr, *cnt = nullptr;
  size_t need = 0;
  if (p.kind == kSplit || p.kind == kChunks)
    need = gqa_split_workspace_bytes(B, H, Sq, D, p.n);
  else if (p.kind == kFlat)
    need = gqa_split_flat_workspace_bytes(B, H, Sq, D, p.n);
  else if (p.kind == kSingle)
    need = gqa_fwd_split_workspace_bytes(B, Hkv, D, p.n);
  // (A captured call gets partials and counters of its own, in Python.)
  if (need > 0 && (capturing() || (ws = stream_buffer(workspaces, dev, stream, need)) == nullptr)) return py::none();
  if (p.kind == kSingle && p.n > 0) {
    const size_t n = gqa_fwd_split_counters_count(B, Hkv, p.n);
    if (capturing() || (cnt = stream_buffer(counters, dev, stream, n * sizeof(int))) == nullptr) return py::none();
  }
  at::Tensor out;
  if (hout.is_none()) {
    out = at::empty(q.sizes(), q.options());
  } else {
    const at::Tensor* po = plain(hout);
    if (po == nullptr || po->sizes() != q.sizes() || po->scalar_type() != q.scalar_type() || po->get_device() != dev ||
        !rows_ready(*po))
      return py::none();
    out = *po;
  }
  at::Tensor lse;
  if (return_lse)
    lse = varlen ? at::empty({q.size(0), H}, q.options().dtype(at::kFloat))
                 : at::empty({B, H, Sq}, q.options().dtype(at::kFloat));
  float* lse_p = return_lse ? lse.data_ptr<float>() : nullptr;
  int64_t qs[4], os[4], ks[4], vs[4];
  if (varlen) {
    const int64_t qv[4] = {0, q.stride(1), q.stride(0), 1}, ov[4] = {0, out.stride(1), out.stride(0), 1};
    std::copy(qv, qv + 4, qs);
    std::copy(ov, ov + 4, os);
  } else {
    strides_of(q, qs);
    strides_of(out, os);
  }
  strides_of(kc, ks);
  strides_of(vc, vs);
  const int b = B, h = H, hkv = Hkv, sq = Sq, d = D, c = causal ? 1 : 0, dt = dtype_code(q), bsz = bs;
  const int ms = max_seq_len, ts = B > 1 ? tab.stride(0) : tab.size(1);
  const float sl2 = scale_log2;
  const int *tp = tab.data_ptr<int>(), *lp = lens.data_ptr<int>();
  const int* qsp = varlen ? qst->data_ptr<int>() : nullptr;
  const int* qlp = varlen ? qln->data_ptr<int>() : nullptr;
  float* wsf = static_cast<float*>(ws);
  const void *qp = q.data_ptr(), *kp = kc.data_ptr(), *vp = vc.data_ptr();
  void* op = out.data_ptr();
  if (p.kind == kFlat) {
    const int rc = gqa_paged_split_flat_launch(qp, qs, kp, ks, vp, vs, tp, ts, lp, qsp, qlp, bsz, ms, op, os, lse_p,
                                               wsf, p.n, b, h, hkv, sq, d, sl2, c, dt, stream);
    if (rc == GQA_E_FLAT) return py::none();
    check_rc(rc, "gqa_paged_split_flat_launch");
  } else if (p.kind == kShort) {
    check_rc(gqa_paged_fwd_short_launch(qp, qs, kp, ks, vp, vs, tp, ts, lp, qsp, qlp, bsz, ms, op, os, lse_p, b, h,
                                        hkv, sq, d, sl2, c, dt, stream), "gqa_paged_fwd_short_launch");
  } else if (p.kind == kChunks) {
    check_rc(gqa_paged_fwd_chunks_launch(qp, qs, kp, ks, vp, vs, tp, ts, lp, qsp, qlp, bsz, ms, op, os, lse_p, wsf,
                                         p.n, b, h, hkv, sq, d, sl2, c, dt, stream), "gqa_paged_fwd_chunks_launch");
  } else if (p.kind == kSingle && p.n > 0) {
    check_rc(gqa_paged_fwd_split_launch(qp, qs, kp, ks, vp, vs, tp, ts, lp, qsp, qlp, bsz, ms, op, os, lse_p, wsf,
                                        static_cast<int*>(cnt), p.n, b, h, hkv, sq, d, sl2, c, dt, stream),
             "gqa_paged_fwd_split_launch");
  } else if (p.kind == kSingle) {
    check_rc(gqa_paged_fwd_launch(qp, qs, kp, ks, vp, vs, tp, ts, lp, qsp, qlp, bsz, ms, op, os, lse_p, b, h, hkv, sq,
                                  d, sl2, c, dt, stream), "gqa_paged_fwd_launch");
  } else {
    check_rc(gqa_paged_split_first_launch(qp, qs, kp, ks, vp, vs, tp, ts, lp, qsp, qlp, bsz, ms, wsf, p.n, b, h, hkv,
                                          sq, d, sl2, c, dt, stream), "gqa_paged_split_first_launch");
    int rc;
    if (varlen)
      rc = gqa_split_reduce_varlen_launch(wsf, p.n, op, os, lse_p, qsp, qlp, b, h, sq, d, dt, stream);
    else if (return_lse)
      rc = gqa_split_reduce_lse_launch(wsf, p.n, op, os, lse_p, b, h, sq, d, dt, stream);
    else
      rc = gqa_split_reduce_launch(wsf, p.n, op, os, b, h, sq, d, dt, stream);
    check_rc(rc, "gqa_split_reduce_launch");
  }
  if (return_lse) return py::make_tuple(out, lse);
  return py::cast(out);
}

// write_kv with its checks; false (nothing launched): Python takes the call.
bool write_kv(const py::handle& hk, const py::handle& hv, const py::handle& hkc, const py::handle& hvc,
              const py::handle& hslots) {
  const at::Tensor *k = plain(hk), *v = plain(hv), *kc = plain(hkc), *vc = plain(hvc), *sl = plain(hslots);
  if (k == nullptr || v == nullptr || kc == nullptr || vc == nullptr || sl == nullptr || modes_active()) return false;
  if (k->dim() != 3 || v->sizes() != k->sizes() || !caches_ready(*kc, *vc) || kc->size(2) != k->size(1) ||
      kc->size(3) != k->size(2) || k->scalar_type() != kc->scalar_type() || v->scalar_type() != k->scalar_type() ||
      sl->scalar_type() != at::kLong || sl->dim() != 1 || sl->size(0) != k->size(0) || !sl->is_contiguous() ||
      !rows_ready(*k) || !rows_ready(*v))
    return false;
  const int64_t dev = k->get_device();
  if (v->get_device() != dev || kc->get_device() != dev || sl->get_device() != dev || c10::hip::current_device() != dev)
    return false;
  cache_write(*k, *v, *kc, *vc, *sl, dtype_code(*k));
  return true;
}

// gqa_kernels.dispatch._list_makespan, step for step (its docstring describes
// the schedules): runs of count[i] items of cost[i], repeated n_rep times.
double list_makespan(const std::vector<double>& cost, const std::vector<int64_t>& count, int64_t n_rep, int64_t cu,
                     bool persistent, int64_t dyn_min) {
  if (cost.size() != count.size()) throw std::invalid_argument("list_makespan: one count per cost");
  int64_t period = 0;
  for (int64_t k : count) {
    if (k < 0) throw std::invalid_argument("list_makespan: negative count");
    period += k;
  }
  const int64_t total = period * n_rep;
  if (total <= 0) return 0.0;
  const int64_t n_wg = std::min(total, cu), q = total / 8, r = total % 8;
  const bool fixed = persistent && total < dyn_min * n_wg;
  const size_t n = static_cast<size_t>(std::max<int64_t>(1, cu / 8));
  std::vector<double> flat, loads;
  if (fixed)
    for (size_t i = 0; i < cost.size(); ++i) flat.insert(flat.end(), static_cast<size_t>(count[i]), cost[i]);
  std::vector<std::array<int64_t, 3>> seen;
  double worst = 0.0;
  for (int64_t x = 0; x < 8; ++x) {
    const int64_t lo = (x * q + std::min(x, r)) % period, cnt = q + (x < r ? 1 : 0), slots = (n_wg - x + 7) >> 3;
    const std::array<int64_t, 3> key{lo, cnt, fixed ? slots : 0};
    if (cnt == 0 || std::find(seen.begin(), seen.end(), key) != seen.end()) continue;
    seen.push_back(key);
    if (fixed) {
      if (slots < 1) throw std::invalid_argument("list_makespan: fewer than eight CUs");
      // Rows of `slots` items dealt left to right, the odd ones right to left.
      loads.assign(static_cast<size_t>(slots), 0.0);
      for (int64_t e = 0; e < cnt; ++e) {
        const int64_t row = e / slots, at = e % slots;
        loads[static_cast<size_t>(row & 1 ? slots - 1 - at : at)] += flat[static_cast<size_t>((lo + e) % period)];
      }
      worst = std::max(worst, *std::max_element(loads.begin(), loads.end()));
      continue;
    }
    // Each item to the least loaded CU; `loads` ascending.  A run on loads
    // within its cost of each other goes round by round.
    loads.assign(n, 0.0);
    size_t i = 0;
    int64_t off = lo;
    while (off >= count[i]) off -= count[i++];
    for (int64_t left = cnt; left > 0;) {
      const double c = cost[i];
      int64_t k = std::min(count[i] - off, left);
      left -= k;
      // (A run goes on over the end of the period, as _slice_runs joins them.)
      for (;;) {
        i = (i + 1) % cost.size();
        off = 0;
        if (left <= 0 || cost[i] != c) break;
        const int64_t more = std::min(count[i], left);
        k += more;
        left -= more;
      }
      while (k > 0) {
        if (loads.back() - loads.front() <= c) {
          const int64_t full = k / static_cast<int64_t>(n), rem = k % static_cast<int64_t>(n);
          if (full > 0)
            for (double& l : loads) l += static_cast<double>(full) * c;
          for (int64_t j = 0; j < rem; ++j) loads[static_cast<size_t>(j)] += c;
          std::rotate(loads.begin(), loads.begin() + rem, loads.end());
          break;
        }
        const double l = loads.front() + c;
        const auto to = std::upper_bound(loads.begin() + 1, loads.end(), l);
        std::move(loads.begin() + 1, to, loads.begin());
        *(to - 1) = l;
        --k;
      }
    }
    worst = std::max(worst, loads.back());
  }
  return worst;
}

// Host ints to an int32 tensor on `device` in one asynchronous copy from
// pinned memory (the caching host allocator keeps the pinned block until the
// copy has run).
at::Tensor ints_to_device(const std::vector<int32_t>& v, int64_t device) {
  const int64_t n = static_cast<int64_t>(v.size());
  at::Tensor host = at::empty({n}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
  std::copy(v.begin(), v.end(), host.data_ptr<int>());
  return host.to(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device)), at::kInt, /*non_blocking=*/true);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "torch-tensor binding of gqa_split_launch (the split-KV decode step)";
  m.def("split_decode", &split_decode, "split-KV decode: first pass and combine through gqa_split_launch",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("ws"), py::arg("splits"), py::arg("causal"),
        py::arg("scale_log2"), py::arg("dtype"), py::arg("return_lse"));
  m.def("split_flat", &split_flat, "flat split-KV forward through gqa_split_flat_launch", py::arg("q"), py::arg("k"),
        py::arg("v"), py::arg("ws"), py::arg("slots"), py::arg("causal"), py::arg("scale_log2"), py::arg("dtype"),
        py::arg("return_lse"));
  m.def("paged_forward", &paged_forward, "paged attention: one of the kernel routes from tensors",
        py::arg("route"), py::arg("q"), py::arg("k_cache"), py::arg("v_cache"), py::arg("block_table"),
        py::arg("table_stride"), py::arg("seq_lens"), py::arg("q_start"), py::arg("q_len"), py::arg("max_seq_len"),
        py::arg("out"), py::arg("lse"), py::arg("ws"), py::arg("counters"), py::arg("splits"), py::arg("batch"),
        py::arg("seq_q"),
        py::arg("scale_log2"), py::arg("causal"), py::arg("dtype"));
  m.def("cache_write", &cache_write, "store new tokens' K/V at their paged cache slots", py::arg("key"),
        py::arg("value"), py::arg("k_cache"), py::arg("v_cache"), py::arg("slot_mapping"), py::arg("dtype"));
  m.def("flash_attn", &flash_attn, "gqa_flash_attn of a planned shape, or None");
  m.def("paged_attn", &paged_attn, "paged_attention of a planned shape on its default route, or None");
  m.def("write_kv", &write_kv, "write_kv with its checks, or False");
  m.def("set_plan", &set_plan, "register the route of a shape");
  m.def("list_makespan", &list_makespan, "run time of a list of items over the CUs (the routing models)");
  m.def("ints_to_device", &ints_to_device, "host ints to an int32 device tensor, asynchronously");
  m.attr("ABI_VERSION") = gqa_abi_version();
}

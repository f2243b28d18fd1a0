// Host side of the operators in native code: a call of recml_amd.hstu_attention (and its autograd form) goes from
// Python through ONE function here to the kernels' C ABI (include/hstu_attn.h).
//
// Why it exists: a small call is bound by its host work.  Checking the arguments and filling the struct field by field
// from Python took 15 us of a call whose kernel takes 8 - 12 (B=4, L=64, H=2, d=32 in fp32: 16.9 us a call), and autograd's
// Python function objects 60 us more per forward and backward.
//
// What it takes: arguments that are ready for the kernels as they are (GPU tensors of one device, unit stride in the
// last axis, int32 lengths and ids, fp32 tables).  Anything else -- a conversion, a copy, an error to report -- comes back
// as None, and the Python side (recml_amd/hstu_ops.py: build_args), which knows every form and every message, runs.

#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <hip/hip_runtime.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/edge.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>

#include <limits>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "hstu_attn.h"
#include "hstu_block.h"

namespace {

using at::Tensor;
using bf16_bits = uint16_t;

void* stream_of(const Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

bool capturing(void* stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing((hipStream_t)stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// ---------------------------------------------------------------------------
// arguments
// ---------------------------------------------------------------------------

// An optional tensor argument: false when it is something that the Python side has to look at.
bool tensor_arg(PyObject* o, Tensor* out) {
  if (o == Py_None) return true;
  if (!THPVariable_Check(o)) return false;
  *out = THPVariable_Unpack(o);
  return true;
}

bool float_arg(PyObject* o, double* out) {
  if (PyFloat_CheckExact(o)) { *out = PyFloat_AS_DOUBLE(o); return true; }
  if (PyLong_CheckExact(o)) {
    *out = PyLong_AsDouble(o);
    if (*out == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
  }
  return false;
}

bool long_arg(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

// Everything of a call but q, k, v, the bias tables and the dense bias (which may carry gradients).
struct Options {
  Tensor seq_lens, seq_offsets, timestamps, q_seg, kv_seg, mask, q_scale, k_scale;
  int64_t max_len = -1;        // -1: not given
  double n = 0.0;              // <= 0: not given (the padded length)
  double alpha = 1.0, bucket_size = 0.301, dropout_p = 0.0;
  int64_t window = -1;
  uint64_t dropout_seed = 0;
  bool causal = true;
  Tensor mask_rows, bias_rows; // copies of the dense operands with rows of whole 16-byte pieces, where the call needs them
};

bool on(const Tensor& t, c10::Device dev) { return t.is_cuda() && t.device() == dev; }

bool plain(const Tensor& t, c10::Device dev, at::ScalarType type) { return on(t, dev) && t.scalar_type() == type && t.is_contiguous(); }

// fp32 [heads, width] or [width] table with heads in {1, H}
bool table(const Tensor& t, c10::Device dev, int64_t H, int64_t* heads, int64_t* width) {
  if (!plain(t, dev, at::kFloat) || t.dim() < 1 || t.dim() > 2) return false;
  *heads = t.dim() == 2 ? t.size(0) : 1;
  *width = t.size(t.dim() - 1);
  return *heads == 1 || *heads == H;
}

// Fills the struct for tensors that are ready as they are; false: the Python side takes the call.
bool fill(HstuAttnFwdArgs& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& pos, const Tensor& ts_tab,
          const Tensor& bias, const Options& o) {
  const auto dev = q.device();
  if (!q.is_cuda() || !on(k, dev) || !on(v, dev) || !on(out, dev)) return false;
  int qk_dtype, v_dtype;
  switch (q.scalar_type()) {
    case at::kFloat: qk_dtype = v_dtype = HSTU_DTYPE_FP32; break;
    case at::kBFloat16: qk_dtype = v_dtype = HSTU_DTYPE_BF16; break;
    case at::kFloat8_e4m3fn: qk_dtype = HSTU_DTYPE_FP8_E4M3FN; v_dtype = HSTU_DTYPE_BF16; break;
    default: return false;
  }
  const auto v_type = v_dtype == HSTU_DTYPE_FP32 ? at::kFloat : at::kBFloat16;
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != v_type || out.scalar_type() != v_type) return false;
  const bool fp8 = qk_dtype == HSTU_DTYPE_FP8_E4M3FN, jagged = q.dim() == 3;
  if (!jagged && q.dim() != 4) return false;
  if (k.dim() != q.dim() || v.dim() != q.dim() || out.dim() != q.dim()) return false;
  const int last = jagged ? 2 : 3, tok = jagged ? 0 : 1;
  if (q.stride(last) != 1 || k.stride(last) != 1 || v.stride(last) != 1 || out.stride(last) != 1) return false;
  const int64_t H = q.size(last - 1), d = q.size(last), d_v = v.size(last);
  if (k.size(last - 1) != H || v.size(last - 1) != H || k.size(last) != d) return false;
  if (out.size(last - 1) != H || out.size(last) != d_v || out.size(tok) != q.size(tok) || (!jagged && out.size(0) != q.size(0))) return false;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.version = HSTU_ATTN_ABI_VERSION;
  a.qk_dtype = qk_dtype;
  a.v_dtype = a.out_dtype = v_dtype;
  int64_t B, L, Lkv;
  if (jagged) {
    const int64_t T = q.size(0);
    if (!o.seq_offsets.defined() || o.max_len < 1 || k.size(0) != T || v.size(0) != T) return false;
    if (!plain(o.seq_offsets, dev, at::kInt) || o.seq_offsets.dim() != 1 || o.seq_offsets.numel() < 1) return false;
    if (o.q_seg.defined() || o.kv_seg.defined()) return false;
    B = o.seq_offsets.numel() - 1;
    L = Lkv = o.max_len;
    a.layout = HSTU_LAYOUT_JAGGED;
    a.total_tokens = T;
    a.seq_offsets = o.seq_offsets.const_data_ptr<int32_t>();
    a.mask_mode = HSTU_MASK_LENGTH;
  } else {
    B = q.size(0);
    L = q.size(1);
    Lkv = k.size(1);
    if (k.size(0) != B || v.size(0) != B || v.size(1) != Lkv || (o.max_len >= 0 && o.max_len != L)) return false;
    a.layout = HSTU_LAYOUT_PADDED;
    if (o.q_seg.defined() != o.kv_seg.defined()) return false;
    if (o.q_seg.defined()) {
      if (o.seq_lens.defined() || !plain(o.q_seg, dev, at::kInt) || !plain(o.kv_seg, dev, at::kInt) || o.q_seg.dim() != 2 || o.kv_seg.dim() != 2 ||
          o.q_seg.size(0) != B || o.q_seg.size(1) != L || o.kv_seg.size(0) != B || o.kv_seg.size(1) != Lkv) return false;
      a.q_segment_ids = o.q_seg.const_data_ptr<int32_t>();
      a.kv_segment_ids = o.kv_seg.const_data_ptr<int32_t>();
      a.mask_mode = HSTU_MASK_SEGMENT;
    } else if (o.seq_lens.defined()) {
      if (!plain(o.seq_lens, dev, at::kInt) || o.seq_lens.dim() != 1 || o.seq_lens.size(0) != B) return false;
      a.seq_lens = o.seq_lens.const_data_ptr<int32_t>();
      a.mask_mode = HSTU_MASK_LENGTH;
    } else {
      a.mask_mode = HSTU_MASK_NONE;
    }
    a.q_stride_b = q.stride(0); a.k_stride_b = k.stride(0); a.v_stride_b = v.stride(0); a.o_stride_b = out.stride(0);
  }
  constexpr int64_t most = std::numeric_limits<int32_t>::max();
  if (B > most || L > most || Lkv > most || H > most) return false;
  a.q = q.const_data_ptr(); a.k = k.const_data_ptr(); a.v = v.const_data_ptr(); a.out = const_cast<void*>(out.const_data_ptr());
  a.q_stride_t = q.stride(tok); a.k_stride_t = k.stride(tok); a.v_stride_t = v.stride(tok); a.o_stride_t = out.stride(tok);
  a.q_stride_h = q.stride(tok + 1); a.k_stride_h = k.stride(tok + 1); a.v_stride_h = v.stride(tok + 1); a.o_stride_h = out.stride(tok + 1);
  a.B = (int32_t)B; a.L = (int32_t)L; a.Lkv = (int32_t)Lkv; a.H = (int32_t)H; a.d_qk = (int32_t)d; a.d_v = (int32_t)d_v;
  if (o.q_scale.defined() || o.k_scale.defined()) {
    if (!fp8) return false;
    for (const Tensor* s : {&o.q_scale, &o.k_scale})
      if (s->defined() && (!plain(*s, dev, at::kFloat) || s->numel() != H)) return false;
    if (o.q_scale.defined()) a.q_scale = o.q_scale.const_data_ptr<float>();
    if (o.k_scale.defined()) a.k_scale = o.k_scale.const_data_ptr<float>();
  }
  a.alpha = (float)o.alpha;
  a.inv_n = (float)(1.0 / (o.n > 0.0 ? o.n : (double)L));
  a.causal = o.causal ? 1 : 0;
  a.window = o.window < 0 ? -1 : (int32_t)(o.window < most ? o.window : most);
  a.dropout_p = (float)o.dropout_p;
  a.dropout_seed = o.dropout_seed;
  if (o.mask.defined()) {
    const Tensor& m = o.mask;
    if (!on(m, dev) || !m.is_contiguous() || (m.scalar_type() != at::kBool && m.scalar_type() != at::kByte) || m.dim() < 2 || m.dim() > 3) return false;
    if (m.size(m.dim() - 2) != L || m.size(m.dim() - 1) != Lkv || (m.dim() == 3 && m.size(0) != B)) return false;
    a.mask = (const uint8_t*)m.const_data_ptr();
    a.mask_batched = m.dim() == 3;
  }
  if (bias.defined()) {
    if (!plain(bias, dev, at::kFloat) || bias.dim() < 2 || bias.dim() > 3) return false;
    if (bias.size(bias.dim() - 2) != L || bias.size(bias.dim() - 1) != Lkv) return false;
    if (bias.dim() == 3 && bias.size(0) != 1 && bias.size(0) != B) return false;
    a.dense_bias = bias.const_data_ptr<float>();
    a.dense_bias_batched = bias.dim() == 3 && B > 1 && bias.size(0) == B;
  }
  int64_t heads, width;
  if (pos.defined()) {
    if (L != Lkv || !table(pos, dev, H, &heads, &width) || width != 2 * L - 1) return false;
    a.pos_tab = pos.const_data_ptr<float>();
    a.pos_heads = (int32_t)heads;
  }
  if (o.timestamps.defined() != ts_tab.defined()) return false;
  if (ts_tab.defined()) {
    const Tensor& ts = o.timestamps;
    if (L != Lkv || !table(ts_tab, dev, H, &heads, &width) || width < 1 || width > most || !plain(ts, dev, at::kLong)) return false;
    if (ts.dim() == 2 && ts.size(0) == B && ts.size(1) == L) a.ts_stride_b = L;
    else if (ts.dim() == 1 && jagged && ts.numel() == q.size(0)) a.ts_stride_b = 0;
    else return false;
    a.ts_tab = ts_tab.const_data_ptr<float>();
    a.ts_heads = (int32_t)heads;
    a.ts = ts.const_data_ptr<int64_t>();
    a.ts_num_buckets = (int32_t)(width - 1);
    a.ts_bucket_size = (float)o.bucket_size;
  }
  return true;
}

// Gives a dense mask or bias whose rows cannot be fetched 16 bytes at a time longer rows, where that is all that keeps the call
// off the matrix-core kernels (B=16, L=1000, H=8, d=64 with gradients: 1.22 ms there, 0.38 on the matrix cores).  The copies are
// left in `o`, for the backward; copies found there are used.
void pad_dense(HstuAttnFwdArgs& a, Options& o, const Tensor& like) {
  if ((!a.mask && !a.dense_bias) || a.qk_dtype != HSTU_DTYPE_BF16 || a.L != a.Lkv) return;
  auto on_mfma = [](const HstuAttnFwdArgs& x) { return !strcmp(hstu_attn_fwd_variant(&x), "hstu_fwd_mfma_bf16"); };
  if (on_mfma(a)) return;
  HstuAttnFwdArgs b = a;
  const bool m = a.mask && (a.Lkv % 16 || ((uintptr_t)a.mask & 15)), d = a.dense_bias && (a.Lkv % 4 || ((uintptr_t)a.dense_bias & 15));
  if (m) { b.mask = (const uint8_t*)256; b.mask_pitch = (a.Lkv + 15) / 16 * 16; }
  if (d) { b.dense_bias = (const float*)256; b.bias_pitch = (a.Lkv + 3) / 4 * 4; }
  if ((!m && !d) || !on_mfma(b)) return;
  auto rows = [&](Tensor& kept, const void* src, int64_t batches, int64_t pitch, int size) {
    if (!kept.defined()) {
      kept = at::empty({batches * a.L * pitch * size}, like.options().dtype(at::kByte).requires_grad(false));
      const int rc = hstu_attn_pad_rows(src, kept.data_ptr(), batches * a.L, a.Lkv, (int32_t)pitch, size, stream_of(like));
      TORCH_CHECK(rc == HSTU_OK, "hstu_attn_pad_rows failed (", rc, "): ", hstu_attn_last_error());
    }
    return kept.const_data_ptr();
  };
  if (m) b.mask = (const uint8_t*)rows(o.mask_rows, a.mask, a.mask_batched ? a.B : 1, b.mask_pitch, 1);
  if (d) b.dense_bias = (const float*)rows(o.bias_rows, a.dense_bias, a.dense_bias_batched ? a.B : 1, b.bias_pitch, 4);
  a = b;
}

Tensor scratch_for(HstuAttnFwdArgs& a, const Tensor& like) {
  const size_t ws = hstu_attn_fwd_workspace_bytes(&a);
  Tensor buf;
  if (ws) {
    buf = at::empty({(int64_t)ws}, like.options().dtype(at::kByte));
    a.workspace = buf.data_ptr();
    a.workspace_bytes = ws;
  }
  return buf;
}

// Whether the device has room for a buffer that a call can do without: in one piece among those that the caching allocator holds, or beside
// them within the process's share.  One that has not makes the allocator wait for the device and give back all that it holds before it fails;
// a training step near the memory's end would do so in every layer's backward.  (Buffers below 64 MB are simply asked for; so are those of
// other allocators, which have no such cache.)
bool has_room(c10::DeviceIndex device, size_t bytes) {
  constexpr size_t SMALL = (size_t)64 << 20, GRAIN = (size_t)2 << 20;
  if (bytes < SMALL) return true;
  try {
    auto* const allocator = c10::hip::HIPCachingAllocator::get();
    if (allocator->name() != "native") return true;
    size_t piece = 1;
    allocator->cacheInfo(device, &piece);
    if (piece >= bytes) return true;
    if (capturing((void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream())) return true;      // (nothing else is asked of the runtime then)
    const c10::DeviceGuard guard(c10::Device(c10::kCUDA, device));
    size_t left = 0, all = 0;
    if (hipMemGetInfo(&left, &all) != hipSuccess) return true;
    const double share = allocator->getMemoryFraction(device) * (double)all -
                         (double)allocator->getDeviceStats(device).reserved_bytes[0].current;
    return left >= bytes + GRAIN && share >= (double)(bytes + GRAIN);
  } catch (const c10::Error&) {
    return true;
  }
}

// The backward's: with room for what its kernels can hand on, or without it where the device has not that much left.  Asked for last, so that
// nothing that the call cannot do without comes after it.
Tensor scratch_for(HstuAttnBwdArgs& b, const Tensor& like) {
  const size_t ws = hstu_attn_bwd_workspace_bytes(&b);
  if (!ws) return Tensor();
  Tensor buf;
  if (has_room(like.device().index(), ws)) {
    try {
      buf = at::empty({(int64_t)ws}, like.options().dtype(at::kByte).requires_grad(false));
    } catch (const c10::OutOfMemoryError&) {
    }
  }
  if (!buf.defined()) {
    const uint32_t flags = b.fwd.flags;
    b.fwd.flags &= ~HSTU_BWD_WRITE_BIAS_GRADIENT;       // (the forward's question knows no flag of the backward's)
    buf = scratch_for(b.fwd, like);
    b.fwd.flags = flags;
    return buf;
  }
  b.fwd.workspace = buf.data_ptr();
  b.fwd.workspace_bytes = ws;
  return buf;
}

// What the calls on one batch share (recml_amd.hstu_ops.AttentionBatch): the workspace, and what it was prepared for.
struct Shared {
  std::string prepared, now;   // signatures: of the workspace as it comes, and of this call (empty: do not share)
  Tensor buf;
  bool reused = false;
};

void sign(std::string& to, const Tensor& t) {
  auto put = [&](int64_t x) { to.append((const char*)&x, sizeof(x)); };
  put(t.defined() ? 1 : 0);
  if (!t.defined()) return;
  put((int64_t)(intptr_t)t.const_data_ptr());
  // (tensors made under torch.inference_mode() carry no version counter)
  put(t.is_inference() ? -1 : (int64_t)t._version());
  put((int64_t)t.scalar_type());
  put(t.dim());
  for (int64_t i = 0; i < t.dim(); ++i) { put(t.size(i)); put(t.stride(i)); }
}

// The forward that fill() has described; false: the Python side takes the call (and reports what is wrong with it).
bool forward(HstuAttnFwdArgs& a, const Tensor& q, const Tensor& pos, const Tensor& ts_tab, const Tensor& bias, Options& o, Shared* shared = nullptr) {
  pad_dense(a, o, q);
  if (!shared) {
    const Tensor buf = scratch_for(a, q);
    return hstu_attn_fwd(&a, stream_of(q)) == HSTU_OK;
  }
  const int64_t ws = (int64_t)hstu_attn_fwd_workspace_bytes(&a);
  shared->now.clear();
  if (ws) {
    // everything the preparation reads or the workspace's layout depends on (segment ids: no sharing)
    if (!o.q_seg.defined()) {
      for (const Tensor* t : std::initializer_list<const Tensor*>{&o.seq_lens, &o.seq_offsets, &o.timestamps, &pos, &ts_tab, &o.mask}) sign(shared->now, *t);
      const int64_t more[] = {a.layout, a.B, a.L, a.Lkv, a.H, a.d_qk, a.d_v, a.total_tokens, a.qk_dtype, a.causal, a.window, bias.defined(), ws};
      shared->now.append((const char*)more, sizeof(more));
      shared->now.append((const char*)&a.ts_bucket_size, sizeof(float));
    }
    if (!shared->buf.defined() || shared->buf.numel() != ws || shared->buf.device() != q.device()) {
      shared->buf = at::empty({ws}, q.options().dtype(at::kByte).requires_grad(false));
      shared->prepared.clear();
    }
    a.workspace = shared->buf.data_ptr();
    a.workspace_bytes = (size_t)ws;
    if (!shared->now.empty() && shared->now == shared->prepared) {
      a.flags |= HSTU_FWD_WORKSPACE_PREPARED;
      shared->reused = true;
    }
  }
  return hstu_attn_fwd(&a, stream_of(q)) == HSTU_OK;
}

Tensor like_output(const Tensor& q, const Tensor& v) {
  auto shape = q.sizes().vec();
  shape.back() = v.size(-1);
  return at::empty(shape, v.options().requires_grad(false));
}

// ---------------------------------------------------------------------------
// autograd
// ---------------------------------------------------------------------------

// dq, dk, dv with the strides of q, k, v.  Slices of one projection get slices of one buffer laid out like it (mirrored
// one by one each would span nearly all of the projection).
void gradient_buffers(const Tensor (&t)[3], Tensor (&g)[3]) {
  bool shared = true;
  int64_t lo = std::numeric_limits<int64_t>::max(), hi = 0, total = 0;
  for (const Tensor& x : t) {
    if (!x.numel() || x.scalar_type() != t[0].scalar_type() || !x.storage().is_alias_of(t[0].storage())) { shared = false; break; }
    int64_t extent = 1;
    for (int64_t i = 0; i < x.dim(); ++i) extent += (x.size(i) - 1) * x.stride(i);
    lo = std::min(lo, x.storage_offset());
    hi = std::max(hi, x.storage_offset() + extent);
    total += x.numel();
  }
  if (shared && hi - lo <= 2 * total) {
    const Tensor buf = at::empty({hi - lo}, t[0].options().requires_grad(false));
    for (int i = 0; i < 3; ++i) g[i] = buf.as_strided(t[i].sizes(), t[i].strides(), t[i].storage_offset() - lo);
    return;
  }
  for (int i = 0; i < 3; ++i) g[i] = at::empty_strided(t[i].sizes(), t[i].strides(), t[i].options().requires_grad(false));
}

struct AttentionBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable q, k, v, pos, ts_tab, bias, mask_rows, bias_rows;
  Options opts;
  bool has_pos = false, has_ts = false, has_bias = false, has_mask_rows = false, has_bias_rows = false;

  std::string name() const override { return "HstuAttentionBackward"; }

  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto* s : {&q, &k, &v, &pos, &ts_tab, &bias, &mask_rows, &bias_rows}) s->reset_data();
    opts = Options();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const at::NoGradGuard no_grad;
    torch::autograd::variable_list result(6);
    if (!grads[0].defined()) return result;
    const Tensor t[3] = {q.unpack(), k.unpack(), v.unpack()};
    const Tensor p = has_pos ? pos.unpack() : Tensor(), tt = has_ts ? ts_tab.unpack() : Tensor(), bs = has_bias ? bias.unpack() : Tensor();
    const c10::DeviceGuard guard(t[0].device());
    const Tensor dout = grads[0].contiguous();
    HstuAttnBwdArgs b;
    memset(&b, 0, sizeof(b));
    b.struct_size = sizeof(b);
    b.version = HSTU_ATTN_ABI_VERSION;
    // (the forward struct's `out` is not read by the backward, which takes dout's strides from it)
    TORCH_CHECK(dout.scalar_type() == t[2].scalar_type() && fill(b.fwd, t[0], t[1], t[2], dout, p, tt, bs, opts),
                "the gradient of hstu_attention's result does not fit the call");
    Options rows = opts;
    if (has_mask_rows) rows.mask_rows = mask_rows.unpack();
    if (has_bias_rows) rows.bias_rows = bias_rows.unpack();
    pad_dense(b.fwd, rows, t[0]);
    Tensor g[3];
    gradient_buffers(t, g);
    b.dout = dout.const_data_ptr();
    b.dq = g[0].data_ptr(); b.dk = g[1].data_ptr(); b.dv = g[2].data_ptr();
    // both tables' gradients when either is wanted; they are added to, so they start as zeros: one buffer, one fill
    const bool want_tables = (has_pos && task_should_compute_output(3)) || (has_ts && task_should_compute_output(4));
    Tensor dpos, dts, dbias;
    if (want_tables) {
      const int64_t np = has_pos ? (p.numel() + 63) / 64 * 64 : 0, nt = has_ts ? tt.numel() : 0;
      const Tensor both = at::zeros({np + nt}, t[0].options().dtype(at::kFloat).requires_grad(false));
      if (has_pos) {
        dpos = both.as_strided(p.sizes(), p.strides(), 0);
        b.dpos_tab = dpos.data_ptr<float>();
      }
      if (has_ts) {
        dts = both.as_strided(tt.sizes(), tt.strides(), np);
        b.dts_tab = dts.data_ptr<float>();
      }
    }
    if (has_bias && task_should_compute_output(5)) {
      dbias = at::empty(bs.sizes(), bs.options().requires_grad(false));
      b.ddense_bias = dbias.data_ptr<float>();
      b.fwd.flags |= HSTU_BWD_WRITE_BIAS_GRADIENT;
    }
    const Tensor scratch = scratch_for(b, t[0]);
    const int rc = hstu_attn_bwd(&b, stream_of(t[0]));
    TORCH_CHECK(rc == HSTU_OK, "hstu_attn_bwd failed (", rc, "): ", hstu_attn_last_error());
    for (int i = 0; i < 3; ++i)
      if (task_should_compute_output(i)) result[i] = g[i];
    if (task_should_compute_output(3)) result[3] = dpos;
    if (task_should_compute_output(4)) result[4] = dts;
    result[5] = dbias;
    return result;
  }
};

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// Whether a tensor carries a forward-mode tangent.  The kernels give none for their results: such a call goes the Python way, whose
// torch steps carry tangents on and whose autograd functions refuse them.
bool dual(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && t->_fw_grad(0).defined()) return true;
  return false;
}

// ---------------------------------------------------------------------------
// block steps
// ---------------------------------------------------------------------------

void block_check(int rc, const char* what) { TORCH_CHECK(rc == HSTU_BLOCK_OK, what, " failed (", rc, "): ", hstu_block_last_error()); }

bool aligned(const Tensor& t) { return ((uintptr_t)t.const_data_ptr() & 15u) == 0; }

// A contiguous, aligned bf16 GPU tensor.
bool ready(const Tensor& t, c10::Device dev) { return t.defined() && plain(t, dev, at::kBFloat16) && aligned(t); }

Tensor fresh(const Tensor& like, at::IntArrayRef shape) { return at::empty(shape, like.options().requires_grad(false)); }

// rows of `width` elements, `stride` apart, as the kernels take them
struct Rows { const void* p; int64_t stride; };

void norm(const Tensor& out, Rows a, Rows u, const Tensor& gamma, const Tensor& beta, int64_t rows, int64_t width, double eps,
          const Tensor& seq_offsets = Tensor(), int64_t L = 0) {
  HstuNormGateArgs g;
  memset(&g, 0, sizeof(g));
  g.struct_size = sizeof(g);
  g.version = HSTU_BLOCK_ABI_VERSION;
  g.rows = rows; g.width = (int32_t)width; g.eps = (float)eps;
  g.a = a.p; g.a_stride = a.stride;
  g.u = u.p; g.u_stride = u.stride;
  g.out = out.data_ptr(); g.out_stride = width;
  g.gamma = gamma.const_data_ptr(); g.beta = beta.const_data_ptr();
  if (seq_offsets.defined()) { g.seq_offsets = seq_offsets.const_data_ptr<int32_t>(); g.L = (int32_t)L; }
  block_check(hstu_norm_gate_fwd(&g, stream_of(out)), "hstu_norm_gate_fwd");
}

// The gradients of norm(): da (and du), and the column sums it returns: those of gamma and beta, fp32 or (rounded) in the parameters' bf16.
struct NormGrad {
  Rows a, u{nullptr, 0}, dout, u_pre{nullptr, 0}, add{nullptr, 0};
  void* da; int64_t da_stride;
  void* du = nullptr; int64_t du_stride = 0;
  Tensor row_map;
};
std::pair<Tensor, Tensor> norm_backward(const NormGrad& n, const Tensor& gamma, const Tensor& beta, int64_t rows, int64_t width, double eps, bool rounded) {
  HstuNormGateBwdArgs g;
  memset(&g, 0, sizeof(g));
  g.struct_size = sizeof(g);
  g.version = HSTU_BLOCK_ABI_VERSION;
  g.rows = rows; g.width = (int32_t)width; g.eps = (float)eps;
  g.a = n.a.p; g.a_stride = n.a.stride; g.u = n.u.p; g.u_stride = n.u.stride; g.dout = n.dout.p; g.dout_stride = n.dout.stride;
  g.da = n.da; g.da_stride = n.da_stride; g.du = n.du; g.du_stride = n.du_stride;
  g.u_pre = n.u_pre.p; g.u_pre_stride = n.u_pre.stride; g.add = n.add.p; g.add_stride = n.add.stride;
  if (n.row_map.defined()) g.row_map = n.row_map.const_data_ptr<int32_t>();
  g.gamma = gamma.const_data_ptr(); g.beta = beta.const_data_ptr();
  const auto sums = gamma.options().dtype(rounded ? at::kBFloat16 : at::kFloat).requires_grad(false);
  const std::pair<Tensor, Tensor> r(at::empty(gamma.sizes(), sums), at::empty(beta.sizes(), sums));
  g.dgamma = (float*)r.first.data_ptr(); g.dbeta = (float*)r.second.data_ptr();
  const int64_t ws = (int64_t)hstu_norm_gate_bwd_workspace_bytes(rows, (int32_t)width);
  const Tensor buf = at::empty({std::max<int64_t>(ws, 16)}, gamma.options().dtype(at::kByte).requires_grad(false));
  g.workspace = buf.data_ptr(); g.workspace_bytes = (size_t)buf.numel();
  block_check((rounded ? hstu_norm_gate_bwd_rounded : hstu_norm_gate_bwd)(&g, stream_of(gamma)), "hstu_norm_gate_bwd");
  return r;
}

void gemm(int op, int64_t M, Rows x, std::initializer_list<const Tensor*> ws, int64_t K, int64_t N, const Tensor& out, const Tensor& bias = Tensor(),
          Rows c = {nullptr, 0}, bool silu = false, const Tensor& pre = Tensor(), Rows y = {nullptr, 0}) {
  HstuGemmArgs g;
  memset(&g, 0, sizeof(g));
  g.struct_size = sizeof(g);
  g.version = HSTU_BLOCK_ABI_VERSION;
  g.op = op; g.activation = silu ? 1 : 0;
  g.M = M; g.N = (int32_t)N; g.K = (int32_t)K;
  g.slabs = (int32_t)ws.size();
  g.x = x.p; g.x_stride = x.stride;
  int i = 0;
  for (const Tensor* w : ws) g.w[i++] = const_cast<void*>(w->const_data_ptr());
  const Tensor& like = **ws.begin();
  Tensor buf;
  if (op == HSTU_GEMM_TN) {
    g.y = y.p; g.y_stride = y.stride;
    const int64_t need = (int64_t)hstu_gemm_workspace_bytes(op, M, g.N, g.K);
    if (need) {
      buf = at::empty({need}, like.options().dtype(at::kByte).requires_grad(false));
      g.workspace = buf.data_ptr();
      g.workspace_bytes = (size_t)need;
    }
  } else {
    g.out = out.data_ptr();
    if (bias.defined()) g.bias = bias.const_data_ptr();
    g.c = c.p; g.c_stride = c.stride;
    if (pre.defined()) g.pre = pre.data_ptr();
  }
  block_check(hstu_gemm(&g, stream_of(like)), "hstu_gemm");
}

// d [M, N] w^T for a weight [K, N] in slabs: the package's kernel for contractions of up to 1024 and small products, torch's
// product (with the slabs put side by side first) for the others.  Microseconds here / there with the concatenation:
//   N = 512 to 512     74 k rows  55 / 66, 131 k  75 / 77        N = 1024 to 256   74 k  61 / 46, 131 k  73 / 68
//   N = 1024 to 1024   6.4 k  25 / 19, 19.2 k  59 / 42
//   N = 2048 to 512    1.6 k  17 / 28, 6.4 k  28 / 27, 19.2 k  50 / 42, 74 k  173 / 185, 131 k  251 / 217
// The library's product is the faster one at most of these, by how much depends on the rows; it is taken where it may save most of
// a step, and kept out of the small calls (one launch here, two there).
Tensor input_gradient(const Tensor& d, std::initializer_list<const Tensor*> ws, int64_t K, int64_t N) {
  const int64_t M = d.size(0), slab = N / (int64_t)ws.size();
  if ((N <= 1024 || 2.0 * (double)M * (double)N * (double)K < 6e9) && (ws.size() == 1 || slab >= 32)) {
    const Tensor out = fresh(d, {M, K});
    gemm(HSTU_GEMM_NT, M, {d.const_data_ptr(), N}, ws, K, N, out);
    return out;
  }
  std::vector<Tensor> parts;
  for (const Tensor* w : ws) parts.push_back(w->view({K, slab}));
  return at::mm(d, (parts.size() == 1 ? parts[0] : at::cat(parts, 1)).t());
}

// A block's parameters in the order Python hands them over.
enum Param { P_IN_G, P_IN_B, P_U, P_Q, P_K, P_V, P_UB, P_QB, P_KB, P_VB, P_ATTN_G, P_ATTN_B, P_OUT, P_OUT_B, P_COUNT };

struct BlockCall {
  int64_t T, D, H, hd, B, L;     // L = 0: packed tokens
  double eps;
  Options opts;
};

bool block_ready(const Tensor& tokens, const Tensor (&p)[P_COUNT], const BlockCall& c, bool training) {
  const auto dev = tokens.device();
  const int64_t W = c.H * c.hd, most = training ? 2048 : 8192;
  if (!ready(tokens, dev) || c.D % 8 || c.hd % 8 || c.D > most || W > most || c.T < 1 || c.T > (1 << 30)) return false;
  for (int i = 0; i < P_COUNT; ++i) {
    const bool optional = (i >= P_UB && i <= P_VB) || i == P_OUT_B;
    if (!p[i].defined()) { if (!optional) return false; continue; }
    if (!ready(p[i], dev)) return false;
  }
  const int64_t n[P_COUNT] = {c.D, c.D, c.D * W, c.D * W, c.D * W, c.D * W, W, W, W, W, W, W, W * c.D, c.D};
  for (int i = 0; i < P_COUNT; ++i)
    if (p[i].defined() && p[i].numel() != n[i]) return false;
  const bool biases = p[P_UB].defined();
  for (int i = P_QB; i <= P_VB; ++i)
    if (p[i].defined() != biases) return false;
  return true;
}

// Whether a block of these sizes and options can be part of one launch for whole blocks.
bool small_shape(const BlockCall& c, const Tensor& ts_tab, const Tensor& bias) {
  const Options& o = c.opts;
  const int64_t L = c.L ? c.L : o.max_len, B = c.L ? c.B : o.seq_offsets.numel() - 1;
  return !ts_tab.defined() && !bias.defined() && !o.mask.defined() && o.dropout_p == 0.0 && o.window < 0 && o.causal && c.D == c.H * c.hd && L <= 64 &&
         c.D <= 64 && B <= 1 << 20 && hstu_block_small_takes((int32_t)B, (int32_t)L, (int32_t)c.H, (int32_t)c.hd, (int32_t)c.D);
}

// Whether its lengths or offsets and its table are as the launch reads them.
bool small_ready(const Tensor& tokens, const BlockCall& c, const Tensor& pos) {
  const Options& o = c.opts;
  const auto dev = tokens.device();
  if (o.timestamps.defined()) return false;
  if (!c.L) {
    if (o.max_len < 1 || o.seq_lens.defined() || !plain(o.seq_offsets, dev, at::kInt) || o.seq_offsets.dim() != 1 || o.seq_offsets.numel() < 1) return false;
  } else if (o.max_len >= 0 || (o.seq_lens.defined() && (!plain(o.seq_lens, dev, at::kInt) || o.seq_lens.dim() != 1 || o.seq_lens.size(0) != c.B))) {
    return false;
  }
  int64_t heads, width;
  return !pos.defined() || (table(pos, dev, c.H, &heads, &width) && width == 2 * (c.L ? c.L : o.max_len) - 1);
}

void fill_small(HstuBlockSmallArgs& a, const Tensor (&p)[P_COUNT], const BlockCall& c, const Tensor& pos) {
  const Options& o = c.opts;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.version = HSTU_BLOCK_ABI_VERSION;
  a.B = (int32_t)(c.L ? c.B : o.seq_offsets.numel() - 1);
  a.L = (int32_t)(c.L ? c.L : o.max_len);
  a.heads = (int32_t)c.H; a.head_dim = (int32_t)c.hd; a.width = (int32_t)c.D;
  a.eps = (float)c.eps; a.alpha = (float)o.alpha; a.inv_n = (float)(1.0 / o.n);
  if (o.seq_lens.defined()) a.seq_lens = o.seq_lens.const_data_ptr<int32_t>();
  if (o.seq_offsets.defined()) a.seq_offsets = o.seq_offsets.const_data_ptr<int32_t>();
  a.in_gamma = p[P_IN_G].const_data_ptr(); a.in_beta = p[P_IN_B].const_data_ptr();
  a.attn_gamma = p[P_ATTN_G].const_data_ptr(); a.attn_beta = p[P_ATTN_B].const_data_ptr();
  for (int i = 0; i < 4; ++i) {
    a.w[i] = p[P_U + i].const_data_ptr();
    if (p[P_UB + i].defined()) a.w_bias[i] = p[P_UB + i].const_data_ptr();
  }
  a.w_out = p[P_OUT].const_data_ptr();
  if (p[P_OUT_B].defined()) a.b_out = p[P_OUT_B].const_data_ptr();
  if (pos.defined()) { a.pos_tab = pos.const_data_ptr<float>(); a.pos_heads = pos.dim() == 2 ? (int32_t)pos.size(0) : 1; }
}

// The block as one launch, where there is one for its shape and options; false: nothing has been done.
bool small_block(Tensor& out, const Tensor& tokens, const Tensor (&p)[P_COUNT], const BlockCall& c, const Tensor& pos, const Tensor& ts_tab, const Tensor& bias) {
  if (!small_shape(c, ts_tab, bias) || !small_ready(tokens, c, pos)) return false;
  HstuBlockSmallArgs a;
  fill_small(a, p, c, pos);
  out = fresh(tokens, tokens.sizes());
  a.tokens = tokens.const_data_ptr(); a.out = out.data_ptr();
  block_check(hstu_block_small_fwd(&a, stream_of(tokens)), "hstu_block_small_fwd");
  return true;
}

// The input norm and the four projections as one launch, where there is one for their sizes; false: nothing has been done.
bool norm_projections(const Tensor& uqkv, const Tensor& tokens, const Tensor (&p)[P_COUNT], int64_t T, int64_t D, int64_t W, double eps) {
  if (T > 0x3fffffff || D > 512 || 4 * W > 1 << 20 || !hstu_norm_gemm_takes(T, (int32_t)(4 * W), (int32_t)D, 4)) return false;
  HstuNormGemmArgs a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.version = HSTU_BLOCK_ABI_VERSION;
  a.M = T; a.N = (int32_t)(4 * W); a.K = (int32_t)D; a.slabs = 4; a.eps = (float)eps;
  a.x = tokens.const_data_ptr(); a.x_stride = D;
  a.gamma = p[P_IN_G].const_data_ptr(); a.beta = p[P_IN_B].const_data_ptr();
  const int order[4] = {P_U, P_Q, P_K, P_V};
  for (int i = 0; i < 4; ++i) a.w[i] = p[order[i]].const_data_ptr();
  a.out = uqkv.data_ptr();
  block_check(hstu_norm_gemm(&a, stream_of(tokens)), "hstu_norm_gemm");
  return true;
}

// slice i of a projection [T, 4, H, hd], shaped as the attention takes it
Tensor projection_slice(const Tensor& uqkv, const BlockCall& c, int i) {
  const int64_t W = c.H * c.hd;
  if (c.L) return uqkv.as_strided({c.B, c.L, c.H, c.hd}, {c.L * 4 * W, 4 * W, c.hd, 1}, uqkv.storage_offset() + i * W);
  return uqkv.as_strided({c.T, c.H, c.hd}, {4 * W, c.hd, 1}, uqkv.storage_offset() + i * W);
}

const bf16_bits* at_column(const Tensor& t, int64_t column) { return (const bf16_bits*)t.const_data_ptr() + column; }

// recml_amd.hstu_block_ops.norm_gate_bwd within the block's backward, on rows that are ready for it.
struct NormOp {
  Tensor da, dgamma, dbeta;
  NormOp(const Tensor& attn, const Tensor& u, const Tensor& gamma, const Tensor& beta, const Tensor& dout, double eps, const Tensor& du_out,
         const Tensor& u_pre, const Tensor& add) {
    const int64_t rows = attn.size(0), W = attn.size(1);
    da = fresh(attn, {rows, W});
    NormGrad n;
    n.a = {attn.const_data_ptr(), attn.stride(0)};
    n.dout = {dout.const_data_ptr(), dout.stride(0)};
    n.da = da.data_ptr(); n.da_stride = W;
    if (u.defined()) {
      n.u = {u.const_data_ptr(), u.stride(0)};
      n.u_pre = {u_pre.const_data_ptr(), u_pre.stride(0)};
      n.du = du_out.data_ptr(); n.du_stride = du_out.stride(0);
    }
    if (add.defined()) n.add = {add.const_data_ptr(), add.stride(0)};
    std::tie(dgamma, dbeta) = norm_backward(n, gamma, beta, rows, W, eps, true);
  }
};

// A tensor kept for the backward, the forward's own intermediates included: this way torch's saved-tensor hooks see it (checkpointing
// and offloading replace it).
torch::autograd::SavedVariable keep(const Tensor& t) { return torch::autograd::SavedVariable(t, false); }

// How far back a block's backward has to go, by what wants a gradient (`wanted(i)`: the i-th of tokens, the parameters, pos, ts_tab).
struct BlockWants {
  bool kernels = false, input, projections, attention, gate;
  template <typename F>
  explicit BlockWants(F&& wanted) {
    bool biases = false;
    for (int i = P_U; i <= P_V; ++i) kernels = kernels || wanted(1 + i);
    for (int i = P_UB; i <= P_VB; ++i) biases = biases || wanted(1 + i);
    input = wanted(0) || wanted(1 + P_IN_G) || wanted(1 + P_IN_B);
    projections = kernels || biases || input;
    attention = projections || wanted(1 + P_COUNT) || wanted(1 + P_COUNT + 1);
    gate = attention || wanted(1 + P_ATTN_G) || wanted(1 + P_ATTN_B);
  }
};

struct BlockBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable tokens, params[P_COUNT], pos, ts_tab;
  bool has[P_COUNT] = {}, has_pos = false, has_ts = false;
  torch::autograd::SavedVariable saved_normed, saved_pre, saved_uqkv, saved_attn, saved_gated;       // of the forward
  BlockCall call;

  std::string name() const override { return "HstuBlockBackward"; }

  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    tokens.reset_data();
    for (auto& p : params) p.reset_data();
    for (auto* x : {&pos, &ts_tab, &saved_normed, &saved_pre, &saved_uqkv, &saved_attn, &saved_gated}) x->reset_data();
    call.opts = Options();
  }

  // Gradients in the order of the edges: tokens, the parameters, pos, ts_tab.  The steps are undone from the output on, as far as a
  // gradient is asked for behind them.
  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const at::NoGradGuard no_grad;
    torch::autograd::variable_list r(1 + P_COUNT + 2);
    if (!grads[0].defined()) return r;
    const BlockWants w([&](int i) { return task_should_compute_output(i); });
    const Tensor x = tokens.unpack();
    const c10::DeviceGuard guard(x.device());
    Tensor p[P_COUNT];
    for (int i = 0; i < P_COUNT; ++i)
      if (has[i]) p[i] = params[i].unpack();
    const int64_t T = call.T, D = call.D, W = call.H * call.hd;
    auto want = [&](int i) { return task_should_compute_output(1 + i); };
    Tensor dout = grads[0].contiguous().view({T, D});
    if (!aligned(dout)) dout = dout.clone();
    // output product
    const Tensor wo = p[P_OUT].view({W, D});
    if (want(P_OUT)) {
      const Tensor g = fresh(p[P_OUT], p[P_OUT].sizes()), gated = saved_gated.unpack();
      gemm(HSTU_GEMM_TN, T, {gated.const_data_ptr(), W}, {&g}, W, D, Tensor(), Tensor(), {nullptr, 0}, false, Tensor(), {dout.const_data_ptr(), D});
      r[1 + P_OUT] = g;
    }
    if (has[P_OUT_B] && want(P_OUT_B)) r[1 + P_OUT_B] = dout.sum(0);
    if (!w.gate) return r;
    // attention norm and gate: du lands in the projection's gradient, already through its SiLU
    const Tensor d_gated = input_gradient(dout, {&wo}, W, D);
    const Tensor pre = saved_pre.unpack(), uqkv = saved_uqkv.unpack(), attn = saved_attn.unpack();
    const Tensor d_uqkv = at::empty_like(uqkv);
    auto rows_of = [&](const Tensor& t, int64_t stride) { return t.as_strided({T, W}, {stride, 1}, t.storage_offset()); };
    const NormOp gate(rows_of(attn, W), rows_of(uqkv, 4 * W), p[P_ATTN_G], p[P_ATTN_B], d_gated, call.eps, rows_of(d_uqkv, 4 * W), rows_of(pre, 4 * W),
                      Tensor());
    if (want(P_ATTN_G)) r[1 + P_ATTN_G] = gate.dgamma;
    if (want(P_ATTN_B)) r[1 + P_ATTN_B] = gate.dbeta;
    if (!w.attention) return r;
    // attention: dq, dk, dv land next to it
    const Tensor d_attn = gate.da.view(attn.sizes());
    const Tensor pt = has_pos ? pos.unpack() : Tensor(), tt = has_ts ? ts_tab.unpack() : Tensor();
    bool through_silu;
    {
      const Tensor q = projection_slice(uqkv, call, 1), k = projection_slice(uqkv, call, 2), v = projection_slice(uqkv, call, 3);
      HstuAttnBwdArgs b;
      memset(&b, 0, sizeof(b));
      b.struct_size = sizeof(b);
      b.version = HSTU_ATTN_ABI_VERSION;
      TORCH_CHECK(fill(b.fwd, q, k, v, d_attn, pt, tt, Tensor(), call.opts), "the block's attention does not fit its own backward");
      b.dout = d_attn.const_data_ptr();
      b.dq = projection_slice(d_uqkv, call, 1).data_ptr();
      b.dk = projection_slice(d_uqkv, call, 2).data_ptr();
      b.dv = projection_slice(d_uqkv, call, 3).data_ptr();
      const bool want_tables = (has_pos && want(P_COUNT)) || (has_ts && want(P_COUNT + 1));
      Tensor dpos, dts;
      if (want_tables) {
        const int64_t np = has_pos ? (pt.numel() + 63) / 64 * 64 : 0, nt = has_ts ? tt.numel() : 0;
        const Tensor both = at::zeros({np + nt}, q.options().dtype(at::kFloat));
        if (has_pos) { dpos = both.as_strided(pt.sizes(), pt.strides(), 0); b.dpos_tab = dpos.data_ptr<float>(); }
        if (has_ts) { dts = both.as_strided(tt.sizes(), tt.strides(), np); b.dts_tab = dts.data_ptr<float>(); }
      }
      const Tensor scratch = scratch_for(b, q);       // (goes by the gradients that are wanted, too)
      // (through the projections' activation on the way, where those kernels run)
      through_silu = w.projections && !strcmp(hstu_attn_bwd_variant(&b), "hstu_bwd_mfma_bf16");
      const int rc = through_silu ? hstu_attn_bwd_silu(&b, at_column(pre, W), at_column(pre, 2 * W), at_column(pre, 3 * W), stream_of(q))
                                  : hstu_attn_bwd(&b, stream_of(q));
      TORCH_CHECK(rc == HSTU_OK, "hstu_attn_bwd failed (", rc, "): ", hstu_attn_last_error());
      if (has_pos && want(P_COUNT)) r[1 + P_COUNT] = dpos;
      if (has_ts && want(P_COUNT + 1)) r[1 + P_COUNT + 1] = dts;
    }
    if (!w.projections) return r;
    if (!through_silu) block_check(hstu_silu_bwd((void*)at_column(d_uqkv, W), 4 * W, at_column(pre, W), 4 * W, T, (int32_t)(3 * W), stream_of(x)), "hstu_silu_bwd");
    // projections
    const Tensor dz = d_uqkv.view({T, 4 * W});
    if (w.kernels) {
      const Tensor gu = fresh(p[P_U], p[P_U].sizes()), gq = fresh(gu, gu.sizes()), gk = fresh(gu, gu.sizes()), gv = fresh(gu, gu.sizes());
      const Tensor normed = saved_normed.unpack();
      gemm(HSTU_GEMM_TN, T, {normed.const_data_ptr(), D}, {&gu, &gq, &gk, &gv}, D, 4 * W, Tensor(), Tensor(), {nullptr, 0}, false, Tensor(),
           {dz.const_data_ptr(), 4 * W});
      r[1 + P_U] = gu; r[1 + P_Q] = gq; r[1 + P_K] = gk; r[1 + P_V] = gv;
    }
    if (has[P_UB] && (want(P_UB) || want(P_QB) || want(P_KB) || want(P_VB))) {
      const Tensor g = dz.sum(0).view({4, call.H, call.hd});
      for (int i = 0; i < 4; ++i) r[1 + P_UB + i] = g[i];
    }
    if (w.input) {
      const Tensor d_normed = input_gradient(dz, {&p[P_U], &p[P_Q], &p[P_K], &p[P_V]}, D, 4 * W);
      // (with the residual's share added)
      const NormOp in(x.view({T, D}), Tensor(), p[P_IN_G], p[P_IN_B], d_normed, call.eps, Tensor(), Tensor(), dout);
      if (want(P_IN_G)) r[1 + P_IN_G] = in.dgamma;
      if (want(P_IN_B)) r[1 + P_IN_B] = in.dbeta;
      if (task_should_compute_output(0)) r[0] = in.da.view(x.sizes());
    }
    return r;
  }
};

// The embedding front end, layer_norm(scale * table[ids] + pos_table[position]).
struct EmbedCall {
  Tensor ids, row_map;           // int64 [B, L]; int32, or undefined: every entry in order
  int64_t T = 0, L = 0;
  double eps = 0.0, scale = 1.0;
  bool training = false;         // the sum rounded step by step, as training has it without the fused kernel
};

void fill_embed(HstuEmbedNormArgs& a, const EmbedCall& c, const Tensor& table, const Tensor& pos_table, const Tensor& gamma, const Tensor& beta) {
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.version = HSTU_BLOCK_ABI_VERSION;
  a.rows = c.T; a.width = (int32_t)table.size(1); a.eps = (float)c.eps; a.scale = (float)c.scale;
  a.ids = c.ids.const_data_ptr<int64_t>();
  a.table = table.const_data_ptr(); a.vocab = table.size(0); a.table_stride = table.stride(0);
  if (pos_table.defined()) { a.pos_table = pos_table.const_data_ptr(); a.n_positions = pos_table.size(0); a.L = (int32_t)c.L; }
  a.gamma = gamma.const_data_ptr(); a.beta = beta.const_data_ptr();
  if (c.row_map.defined()) a.row_map = c.row_map.const_data_ptr<int32_t>();
  a.round_steps = c.training ? 1 : 0;
}

// The gradient of the front end's table [keys, W], or (by position) of its position table, for the gradient `g` of the rows that were
// summed from them.
struct TableGradient {
  int64_t keys, L;
  double scale;
  int by_position;               // as in HstuEmbedGradArgs
};
Tensor table_gradient(const TableGradient& t, const Tensor& g, const Tensor& ids, const Tensor& row_map) {
  const int64_t W = g.size(1);
  const Tensor out = fresh(g, {t.keys, W});
  HstuEmbedGradArgs a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.version = HSTU_BLOCK_ABI_VERSION;
  a.rows = g.size(0); a.keys = t.keys; a.width = (int32_t)W;
  a.scale = (float)t.scale;
  a.g = g.const_data_ptr(); a.g_stride = W;
  if (ids.defined()) a.ids = ids.const_data_ptr<int64_t>();
  if (row_map.defined()) a.row_map = row_map.const_data_ptr<int32_t>();
  a.L = (int32_t)t.L; a.by_position = t.by_position;
  a.out = out.data_ptr();
  const int64_t ws = (int64_t)hstu_embed_grad_workspace_bytes(a.rows, a.keys, a.width);
  const Tensor buf = at::empty({ws}, g.options().dtype(at::kByte));
  a.workspace = buf.data_ptr(); a.workspace_bytes = (size_t)ws;
  block_check(hstu_embed_grad(&a, stream_of(g)), "hstu_embed_grad");
  return out;
}

// Works on the forward's own copies of the gathered rows and their keys: the caller's ids and tables may be refilled or updated
// before it runs.
struct EmbedBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable rows, keys, row_map, gamma, beta;
  bool packed = false;
  int64_t vocab = 0, positions = 0, L = 0;     // positions = 0: no position table
  double eps = 0.0, scale = 1.0;

  std::string name() const override { return "HstuEmbedBackward"; }

  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto* s : {&rows, &keys, &row_map, &gamma, &beta}) s->reset_data();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const at::NoGradGuard no_grad;
    torch::autograd::variable_list r(4);
    if (!grads[0].defined()) return r;
    const Tensor x = rows.unpack(), ids = keys.unpack(), ga = gamma.unpack(), be = beta.unpack(), map = packed ? row_map.unpack() : Tensor();
    const c10::DeviceGuard guard(x.device());
    const int64_t T = x.size(0), W = x.size(1);
    Tensor dout = grads[0].contiguous().view({T, W});
    if (!aligned(dout)) dout = dout.clone();
    const Tensor da = fresh(x, {T, W});
    NormGrad n;
    n.a = {x.const_data_ptr(), W};
    n.dout = {dout.const_data_ptr(), W};
    n.da = da.data_ptr(); n.da_stride = W;
    const auto sums = norm_backward(n, ga, be, T, W, eps, true);
    if (task_should_compute_output(0)) r[0] = table_gradient({vocab, 0, scale, 0}, da, ids, Tensor());
    // (packed rows gather their positions; in a padded batch the table's rows are broadcast over the sequences: one fp32 sum then)
    if (positions && task_should_compute_output(1)) r[1] = table_gradient({positions, L, 1.0, packed ? 1 : 2}, da, Tensor(), map);
    if (task_should_compute_output(2)) r[2] = sums.first;
    if (task_should_compute_output(3)) r[3] = sums.second;
    return r;
  }
};

// The closing norm, from packed tokens to the padded batch (or rows to rows).
struct FinalNormBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable x, gamma, beta, row_map;
  bool packed = false;
  double eps = 0.0;

  std::string name() const override { return "HstuFinalNormBackward"; }

  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto* s : {&x, &gamma, &beta, &row_map}) s->reset_data();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const at::NoGradGuard no_grad;
    torch::autograd::variable_list r(3);
    if (!grads[0].defined()) return r;
    const Tensor a = x.unpack(), ga = gamma.unpack(), be = beta.unpack();
    const c10::DeviceGuard guard(a.device());
    const int64_t W = a.size(-1), rows = a.numel() / W;
    Tensor dout = grads[0].contiguous();
    if (!aligned(dout)) dout = dout.clone();
    const Tensor da = fresh(a, a.sizes());
    NormGrad n;
    n.a = {a.const_data_ptr(), W};
    n.dout = {dout.const_data_ptr(), W};
    n.da = da.data_ptr(); n.da_stride = W;
    if (packed) n.row_map = row_map.unpack();
    const auto sums = norm_backward(n, ga, be, rows, W, eps, true);
    if (task_should_compute_output(0)) r[0] = da;
    if (task_should_compute_output(1)) r[1] = sums.first;
    if (task_should_compute_output(2)) r[2] = sums.second;
    return r;
  }
};

// x [M, K] w [K, N] with gradients, and theirs where they are asked for (create_graph: torch's products then).
struct LinearBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable x, w;

  std::string name() const override { return "HstuLinearBackward"; }

  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x.reset_data();
    w.reset_data();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    torch::autograd::variable_list r(2);
    if (!grads[0].defined()) return r;
    const Tensor a = x.unpack(), b = w.unpack();
    const c10::DeviceGuard guard(a.device());
    if (at::GradMode::is_enabled()) {
      if (task_should_compute_output(0)) r[0] = at::matmul(grads[0], b.t());
      if (task_should_compute_output(1)) r[1] = at::matmul(a.flatten(0, -2).t(), grads[0].flatten(0, -2));
      return r;
    }
    const at::NoGradGuard no_grad;
    const int64_t K = b.size(0), N = b.size(1), M = a.numel() / K;
    Tensor d = grads[0].contiguous().view({M, N});
    if (!aligned(d)) d = d.clone();
    if (task_should_compute_output(0)) r[0] = input_gradient(d, {&b}, K, N).view(a.sizes());
    if (task_should_compute_output(1)) {
      const Tensor g = fresh(b, b.sizes());
      gemm(HSTU_GEMM_TN, M, {a.const_data_ptr(), K}, {&g}, K, N, Tensor(), Tensor(), {nullptr, 0}, false, Tensor(), {d.const_data_ptr(), N});
      r[1] = g;
    }
    return r;
  }
};

// ---------------------------------------------------------------------------
// Python
// ---------------------------------------------------------------------------

// Runs `f`; an exception becomes the Python one of its type (torch.OutOfMemoryError, IndexError, an error of a hook, ...).
template <typename F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  return f();
  END_HANDLE_TH_ERRORS
}

enum Arg { A_Q, A_K, A_V, A_SEQ_LENS, A_SEQ_OFFSETS, A_MAX_LEN, A_N, A_ALPHA, A_CAUSAL, A_POS, A_TS, A_TS_TAB, A_BUCKET, A_QSEG, A_KVSEG, A_WINDOW,
           A_MASK, A_BIAS, A_OUT, A_QSCALE, A_KSCALE, A_DROP_P, A_DROP_SEED, A_GRAD, A_COUNT };

// attention(q, k, v, seq_lens, ..., dropout_seed, differentiable) -> Tensor, or None when the Python side has to take
// the call.  `differentiable`: the result carries gradients for q, k, v, the tables and the dense bias where they want them.
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != A_COUNT) {
    PyErr_Format(PyExc_TypeError, "attention takes %d arguments, got %zd", (int)A_COUNT, count);
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor q, k, v, pos, ts_tab, bias, out;
    Options o;
    for (int i : {A_Q, A_K, A_V})
      if (!THPVariable_Check(args[i])) Py_RETURN_NONE;
    q = THPVariable_Unpack(args[A_Q]);
    k = THPVariable_Unpack(args[A_K]);
    v = THPVariable_Unpack(args[A_V]);
    if (!tensor_arg(args[A_SEQ_LENS], &o.seq_lens) || !tensor_arg(args[A_SEQ_OFFSETS], &o.seq_offsets) || !tensor_arg(args[A_POS], &pos) ||
        !tensor_arg(args[A_TS], &o.timestamps) || !tensor_arg(args[A_TS_TAB], &ts_tab) || !tensor_arg(args[A_QSEG], &o.q_seg) ||
        !tensor_arg(args[A_KVSEG], &o.kv_seg) || !tensor_arg(args[A_MASK], &o.mask) || !tensor_arg(args[A_BIAS], &bias) ||
        !tensor_arg(args[A_OUT], &out) || !tensor_arg(args[A_QSCALE], &o.q_scale) || !tensor_arg(args[A_KSCALE], &o.k_scale)) Py_RETURN_NONE;
    if (args[A_MAX_LEN] != Py_None && (!long_arg(args[A_MAX_LEN], &o.max_len) || o.max_len < 1)) Py_RETURN_NONE;
    if (args[A_N] != Py_None && (!float_arg(args[A_N], &o.n) || !(o.n > 0.0))) Py_RETURN_NONE;
    if (args[A_WINDOW] != Py_None && (!long_arg(args[A_WINDOW], &o.window) || o.window < 0)) Py_RETURN_NONE;
    if (!float_arg(args[A_ALPHA], &o.alpha) || !float_arg(args[A_BUCKET], &o.bucket_size) || !float_arg(args[A_DROP_P], &o.dropout_p)) Py_RETURN_NONE;
    if (!(o.dropout_p >= 0.0 && o.dropout_p < 1.0) || !PyLong_CheckExact(args[A_DROP_SEED])) Py_RETURN_NONE;
    o.dropout_seed = PyLong_AsUnsignedLongLongMask(args[A_DROP_SEED]);
    if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
    const int causal = PyObject_IsTrue(args[A_CAUSAL]);
    if (causal < 0) return nullptr;
    o.causal = causal != 0;
    const bool graph = args[A_GRAD] == Py_True && wants_grad({&q, &k, &v, &pos, &ts_tab, &bias});
    if (args[A_GRAD] == Py_True && dual({&q, &k, &v, &pos, &ts_tab, &bias})) Py_RETURN_NONE;
    if (!q.is_cuda() || q.dim() < 1 || v.dim() != q.dim() || (graph && (out.defined() || q.scalar_type() == at::kFloat8_e4m3fn))) Py_RETURN_NONE;
    bool ok;
    {
      PyThreadState* const saved = PyEval_SaveThread();
      try {
        const c10::DeviceGuard guard(q.device());
        const at::NoGradGuard no_grad;
        if (!out.defined()) out = like_output(q, v);
        HstuAttnFwdArgs a;
        ok = fill(a, q, k, v, out, pos, ts_tab, bias, o) && forward(a, q, pos, ts_tab, bias, o);
      } catch (...) {
        PyEval_RestoreThread(saved);
        throw;
      }
      PyEval_RestoreThread(saved);
    }
    if (!ok) Py_RETURN_NONE;
    if (graph) {
      auto node = std::shared_ptr<AttentionBackward>(new AttentionBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(q, k, v, pos, ts_tab, bias));
      node->q = torch::autograd::SavedVariable(q, false);
      node->k = torch::autograd::SavedVariable(k, false);
      node->v = torch::autograd::SavedVariable(v, false);
      node->has_pos = pos.defined();
      node->has_ts = ts_tab.defined();
      node->has_bias = bias.defined();
      if (node->has_pos) node->pos = torch::autograd::SavedVariable(pos, false);
      if (node->has_ts) node->ts_tab = torch::autograd::SavedVariable(ts_tab, false);
      if (node->has_bias) node->bias = torch::autograd::SavedVariable(bias, false);
      if ((node->has_mask_rows = o.mask_rows.defined())) node->mask_rows = torch::autograd::SavedVariable(o.mask_rows, false);
      if ((node->has_bias_rows = o.bias_rows.defined())) node->bias_rows = torch::autograd::SavedVariable(o.bias_rows, false);
      o.mask_rows = o.bias_rows = Tensor();
      node->opts = std::move(o);
      torch::autograd::set_history(out, node);
    }
    return THPVariable_Wrap(std::move(out));
  });
}

// Runs `f` without the interpreter's lock, on the tensor's device, outside of any graph.
template <typename F>
auto without_lock(const Tensor& t, F&& f) {
  struct Release {
    PyThreadState* saved = PyEval_SaveThread();
    ~Release() { PyEval_RestoreThread(saved); }
  } release;
  const c10::DeviceGuard guard(t.device());
  const at::NoGradGuard no_grad;
  return f();
}


// block(tokens [.., D], params, heads, head_dim, eps, alpha, n, seq_lens, seq_offsets, max_len, pos, timestamps, ts_tab, mask, bias,
//       dropout_p, dropout_seed, prepared, workspace, differentiable) -> (out, signature, workspace, reused) or None
// Padded tokens [B, L, D], or packed ones [T, D] with seq_offsets.
PyObject* block(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 20) {
    PyErr_SetString(PyExc_TypeError, "block takes 20 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor tokens, p[P_COUNT], pos, ts_tab, bias;
    BlockCall c;
    Options& o = c.opts;
    if (!tensor_arg(a[0], &tokens) || !tokens.defined() || !PyTuple_CheckExact(a[1]) || PyTuple_GET_SIZE(a[1]) != P_COUNT) Py_RETURN_NONE;
    for (int i = 0; i < P_COUNT; ++i)
      if (!tensor_arg(PyTuple_GET_ITEM(a[1], i), &p[i])) Py_RETURN_NONE;
    if (!long_arg(a[2], &c.H) || !long_arg(a[3], &c.hd) || !float_arg(a[4], &c.eps) || !float_arg(a[5], &o.alpha) || !float_arg(a[6], &o.n) || !(o.n > 0.0))
      Py_RETURN_NONE;
    if (!tensor_arg(a[7], &o.seq_lens) || !tensor_arg(a[8], &o.seq_offsets) || (a[9] != Py_None && !long_arg(a[9], &o.max_len)) ||
        !tensor_arg(a[10], &pos) || !tensor_arg(a[11], &o.timestamps) || !tensor_arg(a[12], &ts_tab) || !tensor_arg(a[13], &o.mask) ||
        !tensor_arg(a[14], &bias) || !float_arg(a[15], &o.dropout_p) || !PyLong_CheckExact(a[16])) Py_RETURN_NONE;
    o.dropout_seed = PyLong_AsUnsignedLongLongMask(a[16]);
    if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
    o.causal = !o.mask.defined();
    Shared shared;
    const bool share = a[17] != Py_False;          // False: the caller keeps nothing
    if (PyBytes_CheckExact(a[17])) shared.prepared.assign(PyBytes_AS_STRING(a[17]), (size_t)PyBytes_GET_SIZE(a[17]));
    if (!tensor_arg(a[18], &shared.buf)) Py_RETURN_NONE;
    if (!tokens.is_cuda() || tokens.dim() != (o.seq_offsets.defined() ? 2 : 3)) Py_RETURN_NONE;
    c.D = tokens.size(-1);
    c.B = tokens.dim() == 3 ? tokens.size(0) : 0;
    c.L = tokens.dim() == 3 ? tokens.size(1) : 0;
    c.T = tokens.dim() == 3 ? c.B * c.L : tokens.size(0);
    const bool graph = a[19] == Py_True && [&] {
      if (!at::GradMode::is_enabled()) return false;
      bool any = tokens.requires_grad();
      for (const Tensor& t : p) any = any || (t.defined() && t.requires_grad());
      for (const Tensor* t : {&pos, &ts_tab, &bias}) any = any || (t->defined() && t->requires_grad());
      return any;
    }();
    if ((graph && (o.mask.defined() || bias.defined())) || !block_ready(tokens, p, c, graph)) Py_RETURN_NONE;
    for (const Tensor& t : p)
      if (dual({&t})) Py_RETURN_NONE;
    if (dual({&tokens, &pos, &ts_tab, &bias})) Py_RETURN_NONE;
    Tensor out, normed, pre, uqkv, attn, gated;
    const bool ok = without_lock(tokens, [&] {
      const int64_t T = c.T, D = c.D, W = c.H * c.hd;
      if (!graph && small_block(out, tokens, p, c, pos, ts_tab, bias)) return true;
      uqkv = fresh(tokens, {T, 4, c.H, c.hd});
      if (c.L) attn = fresh(tokens, {c.B, c.L, c.H, c.hd});
      else attn = fresh(tokens, {T, c.H, c.hd});
      // (a call whose attention the Python side has to take is found here, before any of its work)
      HstuAttnFwdArgs a;
      const Tensor q = projection_slice(uqkv, c, 1);
      if (!fill(a, q, projection_slice(uqkv, c, 2), projection_slice(uqkv, c, 3), attn, pos, ts_tab, bias, o)) return false;
      if (graph || p[P_UB].defined() || !norm_projections(uqkv, tokens, p, T, D, W, c.eps)) {
        normed = fresh(tokens, {T, D});
        norm(normed, {tokens.const_data_ptr(), D}, {nullptr, 0}, p[P_IN_G], p[P_IN_B], T, D, c.eps);
        if (graph) pre = at::empty_like(uqkv);
        Tensor pb;
        if (p[P_UB].defined()) pb = at::cat({p[P_UB].view({W}), p[P_QB].view({W}), p[P_KB].view({W}), p[P_VB].view({W})});
        gemm(HSTU_GEMM_NN, T, {normed.const_data_ptr(), D}, {&p[P_U], &p[P_Q], &p[P_K], &p[P_V]}, D, 4 * W, uqkv, pb, {nullptr, 0}, true, pre);
      }
      if (!forward(a, q, pos, ts_tab, bias, o, share ? &shared : nullptr)) return false;
      gated = fresh(tokens, {T, W});
      norm(gated, {attn.const_data_ptr(), W}, {uqkv.const_data_ptr(), 4 * W}, p[P_ATTN_G], p[P_ATTN_B], T, W, c.eps);
      out = fresh(tokens, tokens.sizes());
      gemm(HSTU_GEMM_NN, T, {gated.const_data_ptr(), W}, {&p[P_OUT]}, W, D, out, p[P_OUT_B], {tokens.const_data_ptr(), D});
      return true;
    });
    if (!ok) Py_RETURN_NONE;
    if (graph) {
      auto node = std::shared_ptr<BlockBackward>(new BlockBackward(), torch::autograd::deleteNode);
      torch::autograd::edge_list edges;
      auto edge = [&](const Tensor& t) { edges.push_back(t.defined() ? torch::autograd::impl::gradient_edge(t) : torch::autograd::Edge()); };
      edge(tokens);
      for (const Tensor& t : p) edge(t);
      edge(pos);
      edge(ts_tab);
      node->set_next_edges(std::move(edges));
      node->tokens = keep(tokens);
      for (int i = 0; i < P_COUNT; ++i)
        if ((node->has[i] = p[i].defined())) node->params[i] = keep(p[i]);
      if ((node->has_pos = pos.defined())) node->pos = keep(pos);
      if ((node->has_ts = ts_tab.defined())) node->ts_tab = keep(ts_tab);
      // (only what the gradients asked for read)
      auto wanted = [&](int i) {
        const Tensor& t = i == 0 ? tokens : i <= P_COUNT ? p[i - 1] : i == P_COUNT + 1 ? pos : ts_tab;
        return t.defined() && t.requires_grad();
      };
      const BlockWants w(wanted);
      if (w.kernels) node->saved_normed = keep(normed);
      if (w.gate) {
        node->saved_pre = keep(pre);
        node->saved_uqkv = keep(uqkv);
        node->saved_attn = keep(attn);
      }
      if (wanted(1 + P_OUT)) node->saved_gated = keep(gated);
      node->call = std::move(c);
      torch::autograd::set_history(out, node);
    }
    PyObject* const sig = PyBytes_FromStringAndSize(shared.now.data(), (Py_ssize_t)shared.now.size());
    PyObject* const buf = shared.buf.defined() ? THPVariable_Wrap(shared.buf) : (Py_INCREF(Py_None), Py_None);
    return Py_BuildValue("(NNNO)", THPVariable_Wrap(std::move(out)), sig, buf, shared.reused ? Py_True : Py_False);
  });
}

// blocks(tokens [.., D], (params, ...), heads, head_dim, eps, alpha, n, seq_lens, seq_offsets, max_len, pos, end_gamma, end_beta, end_eps) -> out
// or None: several blocks one behind the other as one launch (a launch for every HSTU_BLOCK_SMALL_STACK of them), and with end_gamma a layer
// norm behind the last.  Where there is no such launch, or a gradient is asked for, the blocks are called one by one.
PyObject* blocks(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 14) {
    PyErr_SetString(PyExc_TypeError, "blocks takes 14 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor tokens, pos, end_gamma, end_beta;
    BlockCall c;
    Options& o = c.opts;
    double end_eps;
    if (!tensor_arg(a[0], &tokens) || !tokens.defined() || !PyTuple_CheckExact(a[1]) || !long_arg(a[2], &c.H) || !long_arg(a[3], &c.hd) ||
        !float_arg(a[4], &c.eps) || !float_arg(a[5], &o.alpha) || !float_arg(a[6], &o.n) || !(o.n > 0.0) || !tensor_arg(a[7], &o.seq_lens) ||
        !tensor_arg(a[8], &o.seq_offsets) || (a[9] != Py_None && !long_arg(a[9], &o.max_len)) || !tensor_arg(a[10], &pos) ||
        !tensor_arg(a[11], &end_gamma) || !tensor_arg(a[12], &end_beta) || !float_arg(a[13], &end_eps)) Py_RETURN_NONE;
    const int64_t n = PyTuple_GET_SIZE(a[1]);
    if (n < 1 || !tokens.is_cuda() || tokens.dim() != (o.seq_offsets.defined() ? 2 : 3)) Py_RETURN_NONE;
    o.causal = true;
    c.D = tokens.size(-1);
    c.B = tokens.dim() == 3 ? tokens.size(0) : 0;
    c.L = tokens.dim() == 3 ? tokens.size(1) : 0;
    c.T = tokens.dim() == 3 ? c.B * c.L : tokens.size(0);
    if (!small_shape(c, Tensor(), Tensor()) || !small_ready(tokens, c, pos)) Py_RETURN_NONE;
    const auto dev = tokens.device();
    if (end_gamma.defined() && (!ready(end_gamma, dev) || !end_beta.defined() || !ready(end_beta, dev) || end_gamma.numel() != c.D || end_beta.numel() != c.D))
      Py_RETURN_NONE;
    auto differentiates = [](const Tensor& t) { return wants_grad({&t}) || dual({&t}); };
    if (differentiates(tokens) || differentiates(pos) || differentiates(end_gamma) || differentiates(end_beta)) Py_RETURN_NONE;
    std::vector<HstuBlockSmallArgs> args((size_t)n);
    for (int64_t i = 0; i < n; ++i) {
      Tensor p[P_COUNT];
      PyObject* const own = PyTuple_GET_ITEM(a[1], i);
      if (!PyTuple_CheckExact(own) || PyTuple_GET_SIZE(own) != P_COUNT) Py_RETURN_NONE;
      for (int j = 0; j < P_COUNT; ++j)
        if (!tensor_arg(PyTuple_GET_ITEM(own, j), &p[j]) || differentiates(p[j])) Py_RETURN_NONE;
      if (!block_ready(tokens, p, c, false)) Py_RETURN_NONE;
      fill_small(args[(size_t)i], p, c, pos);        // (the caller's tuples keep the parameters)
    }
    Tensor out;
    without_lock(tokens, [&] {
      const void* from = tokens.const_data_ptr();
      for (int64_t i = 0; i < n; i += HSTU_BLOCK_SMALL_STACK) {
        const int64_t m = std::min<int64_t>(n - i, HSTU_BLOCK_SMALL_STACK);
        const bool last = i + m == n;
        // (a launch in between: in place, its workgroups read and write rows of their own sequence only)
        if (i == 0) out = fresh(tokens, tokens.sizes());
        args[(size_t)i].tokens = from;
        args[(size_t)(i + m - 1)].out = out.data_ptr();
        block_check(hstu_block_small_stack_fwd(&args[(size_t)i], (int32_t)m, last && end_gamma.defined() ? end_gamma.const_data_ptr() : nullptr,
                                               last && end_gamma.defined() ? end_beta.const_data_ptr() : nullptr, (float)end_eps, stream_of(tokens)),
                    "hstu_block_small_stack_fwd");
        from = out.const_data_ptr();
      }
      return true;
    });
    return THPVariable_Wrap(std::move(out));
  });
}

// norm_gate_bwd(attn, u, gamma, beta, dout, eps, du_out, u_pre, add) -> (d_attn, d_u, d_gamma, d_beta) or None
// (recml_amd.hstu_block_ops.norm_gate_bwd on 2-d rows that are ready as they are)
PyObject* norm_gate_bwd(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 9) {
    PyErr_SetString(PyExc_TypeError, "norm_gate_bwd takes 9 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor attn, u, gamma, beta, dout, du, u_pre, add;
    double eps;
    if (!tensor_arg(a[0], &attn) || !tensor_arg(a[1], &u) || !tensor_arg(a[2], &gamma) || !tensor_arg(a[3], &beta) || !tensor_arg(a[4], &dout) ||
        !float_arg(a[5], &eps) || !tensor_arg(a[6], &du) || !tensor_arg(a[7], &u_pre) || !tensor_arg(a[8], &add)) Py_RETURN_NONE;
    if (!attn.defined() || !attn.is_cuda() || attn.dim() != 2) Py_RETURN_NONE;
    const auto dev = attn.device();
    const int64_t rows = attn.size(0), W = attn.size(1);
    auto fits = [&](const Tensor& t) {
      return on(t, dev) && t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.size(0) == rows && t.size(1) == W && t.stride(1) == 1 && aligned(t);
    };
    if (W % 8 || W < 8 || W > 2048 || !fits(attn) || !dout.defined() || !fits(dout) || !ready(gamma, dev) || !ready(beta, dev) || gamma.numel() != W ||
        beta.numel() != W) Py_RETURN_NONE;
    for (const Tensor* t : {&u, &du, &u_pre, &add})
      if (t->defined() && !fits(*t)) Py_RETURN_NONE;
    if ((du.defined() || u_pre.defined()) && !u.defined()) Py_RETURN_NONE;
    Tensor da;
    std::pair<Tensor, Tensor> sums;
    without_lock(attn, [&] {
      da = fresh(attn, {rows, W});
      if (u.defined() && !du.defined()) du = fresh(attn, {rows, W});
      NormGrad n;
      n.a = {attn.const_data_ptr(), attn.stride(0)};
      n.dout = {dout.const_data_ptr(), dout.stride(0)};
      n.da = da.data_ptr(); n.da_stride = W;
      if (u.defined()) {
        n.u = {u.const_data_ptr(), u.stride(0)};
        n.du = du.data_ptr(); n.du_stride = du.stride(0);
      }
      if (u_pre.defined()) n.u_pre = {u_pre.const_data_ptr(), u_pre.stride(0)};
      if (add.defined()) n.add = {add.const_data_ptr(), add.stride(0)};
      sums = norm_backward(n, gamma, beta, rows, W, eps, false);
      return true;
    });
    return Py_BuildValue("(NNNN)", THPVariable_Wrap(da), du.defined() ? THPVariable_Wrap(du) : (Py_INCREF(Py_None), Py_None),
                         THPVariable_Wrap(sums.first.view({W})), THPVariable_Wrap(sums.second.view({W})));
  });
}

// A word in pinned host memory that a kernel writes, and the event behind that kernel.
struct Word {
  Tensor host;
  hipEvent_t done = nullptr;
  explicit Word(const Tensor& like) {
    host = at::empty({1}, like.options().dtype(at::kInt).device(at::kCPU).pinned_memory(true).requires_grad(false));
    *host.data_ptr<int32_t>() = 0;
    TORCH_CHECK(hipEventCreateWithFlags(&done, hipEventDisableTiming) == hipSuccess, "hipEventCreate failed");
  }
  Word(const Word&) = delete;
  void record(void* stream) { TORCH_CHECK(hipEventRecord(done, (hipStream_t)stream) == hipSuccess, "hipEventRecord failed"); }
  int32_t wait() {
    TORCH_CHECK(hipEventSynchronize(done) == hipSuccess, "hipEventSynchronize failed");
    return *(volatile int32_t*)host.data_ptr<int32_t>();
  }
  ~Word() {
    // (the word must not go back to the pool while the kernel may still write it)
    if (done) {
      (void)hipEventSynchronize(done);
      (void)hipEventDestroy(done);
    }
  }
};

void drop_word(PyObject* capsule) { delete (Word*)PyCapsule_GetPointer(capsule, "recml_amd.word"); }

// Hands a word over to Python as a ticket: raised(ticket) says whether its kernel raised it.
PyObject* ticket_of(std::unique_ptr<Word> word) {
  PyObject* const capsule = PyCapsule_New(word.get(), "recml_amd.word", drop_word);
  if (capsule) word.release();
  return capsule;
}

PyObject* raised(PyObject*, PyObject* ticket) {
  return guarded([&]() -> PyObject* {
    Word* const word = (Word*)PyCapsule_GetPointer(ticket, "recml_amd.word");
    if (!word) return nullptr;
    int32_t value;
    Py_BEGIN_ALLOW_THREADS
    value = word->wait();
    Py_END_ALLOW_THREADS
    return PyBool_FromLong(value != 0);
  });
}

// Whether hstu_mask_lengths reads this mask as it is.
bool byte_mask(const Tensor& mask) {
  return mask.is_cuda() && mask.dim() == 2 && mask.size(0) >= 1 && mask.size(1) >= 1 && mask.is_contiguous() &&
         (mask.scalar_type() == at::kBool || mask.scalar_type() == at::kByte) && mask.numel() <= 0x7fffffff;
}

// embed(ids, table, pos_table, gamma, beta, eps, scale, row_map, tokens, differentiable, mask) -> (rows [tokens, D] (or shaped like ids), ticket),
// with a mask shaped like ids (rows, ticket, lengths, the lengths' ticket: as from mask_lengths, in the same launch), or None.  Without gradients indices are clamped into their tables and the ticket is None; with them they are taken as torch's indexing
// takes them, and raised(ticket) says that one lay outside.  (A captured step has no ticket: nobody can ask while it is captured.)
PyObject* embed(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 11) {
    PyErr_SetString(PyExc_TypeError, "embed takes 11 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    EmbedCall c;
    Tensor table, pos_table, gamma, beta, mask;
    if (!tensor_arg(a[10], &mask)) Py_RETURN_NONE;
    if (!tensor_arg(a[0], &c.ids) || !tensor_arg(a[1], &table) || !tensor_arg(a[2], &pos_table) || !tensor_arg(a[3], &gamma) || !tensor_arg(a[4], &beta) ||
        !float_arg(a[5], &c.eps) || !float_arg(a[6], &c.scale) || !tensor_arg(a[7], &c.row_map) || !long_arg(a[8], &c.T)) Py_RETURN_NONE;
    if (!c.ids.defined() || !table.defined() || !table.is_cuda() || dual({&table, &pos_table, &gamma, &beta})) Py_RETURN_NONE;
    const auto dev = table.device();
    if (!plain(c.ids, dev, at::kLong) || c.ids.dim() != 2 || !ready(table, dev) || table.dim() != 2 || !ready(gamma, dev) || !ready(beta, dev) ||
        (pos_table.defined() && (!ready(pos_table, dev) || pos_table.dim() != 2 || pos_table.size(1) != table.size(1)))) Py_RETURN_NONE;
    const int64_t D = table.size(1);
    c.L = c.ids.size(1);
    const bool packed = c.row_map.defined();
    // (the map's entries index ids: one with more entries is another batch's)
    if (packed && (!plain(c.row_map, dev, at::kInt) || c.row_map.numel() < c.T || c.row_map.numel() > c.ids.numel())) Py_RETURN_NONE;
    if (mask.defined() && (packed || !byte_mask(mask) || mask.device() != dev || mask.sizes() != c.ids.sizes() || capturing(stream_of(table)))) Py_RETURN_NONE;
    if (!packed) c.T = c.ids.numel();
    const bool graph = a[9] == Py_True && wants_grad({&table, &pos_table, &gamma, &beta});
    // (a padded batch longer than the position table: torch's addition reports it)
    if (graph && !packed && pos_table.defined() && pos_table.size(0) < c.L) Py_RETURN_NONE;
    c.training = graph;
    if (D % 8 || D > (graph ? 2048 : 8192) || c.T < 1 || c.L < 1 || gamma.numel() != D || beta.numel() != D || c.ids.numel() > (1 << 30) ||
        (graph && (table.size(0) > (1 << 30)))) Py_RETURN_NONE;
    Tensor out, sums, keys, lens;
    std::unique_ptr<Word> outside, bad;
    without_lock(table, [&] {
      out = packed ? fresh(table, {c.T, D}) : fresh(table, {c.ids.size(0), c.L, D});
      HstuEmbedNormArgs e;
      fill_embed(e, c, table, pos_table, gamma, beta);
      e.out = out.data_ptr();
      if (graph) {
        sums = fresh(table, {c.T, D});
        keys = at::empty({c.T}, c.ids.options());
        e.sums = sums.data_ptr();
        e.keys = keys.data_ptr<int64_t>();
        if (!capturing(stream_of(table))) {
          outside = std::make_unique<Word>(table);
          e.outside = outside->host.data_ptr<int32_t>();
        }
      }
      if (mask.defined()) {
        lens = at::empty({mask.size(0)}, mask.options().dtype(at::kInt));
        bad = std::make_unique<Word>(mask);
      }
      block_check(hstu_embed_norm_mask_fwd(&e, mask.defined() ? (const uint8_t*)mask.const_data_ptr() : nullptr, (int32_t)c.ids.size(0), (int32_t)c.L,
                                           bad ? lens.data_ptr<int32_t>() : nullptr, bad ? bad->host.data_ptr<int32_t>() : nullptr, stream_of(table)),
                  "hstu_embed_norm_fwd");
      if (outside) outside->record(stream_of(table));
      if (bad) bad->record(stream_of(table));
      return true;
    });
    if (graph) {
      auto node = std::shared_ptr<EmbedBackward>(new EmbedBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(table, pos_table, gamma, beta));
      node->rows = keep(sums);
      node->keys = keep(keys);
      if ((node->packed = packed)) node->row_map = keep(c.row_map);
      node->gamma = keep(gamma);
      node->beta = keep(beta);
      node->vocab = table.size(0);
      node->positions = pos_table.defined() ? pos_table.size(0) : 0;
      node->L = c.L;
      node->eps = c.eps;
      node->scale = c.scale;
      torch::autograd::set_history(out, node);
    }
    PyObject* const ticket = outside ? ticket_of(std::move(outside)) : (Py_INCREF(Py_None), Py_None);
    if (!ticket || !bad) return ticket ? Py_BuildValue("(NN)", THPVariable_Wrap(std::move(out)), ticket) : nullptr;
    PyObject* const end = ticket_of(std::move(bad));
    if (!end) {
      Py_DECREF(ticket);
      return nullptr;
    }
    return Py_BuildValue("(NNNN)", THPVariable_Wrap(std::move(out)), ticket, THPVariable_Wrap(std::move(lens)), end);
  });
}

// final_norm(x, gamma, beta, eps, seq_offsets, row_map, batch, length, differentiable): layer_norm(x), rows to rows, or with
// seq_offsets from packed rows to the padded batch [batch, length, D] with zeros behind each sequence; or None
PyObject* final_norm(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 9) {
    PyErr_SetString(PyExc_TypeError, "final_norm takes 9 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor x, gamma, beta, seq_offsets, row_map;
    double eps;
    int64_t B, L;
    if (!tensor_arg(a[0], &x) || !tensor_arg(a[1], &gamma) || !tensor_arg(a[2], &beta) || !float_arg(a[3], &eps) || !tensor_arg(a[4], &seq_offsets) ||
        !tensor_arg(a[5], &row_map) || !long_arg(a[6], &B) || !long_arg(a[7], &L)) Py_RETURN_NONE;
    if (!x.defined() || !x.is_cuda() || x.dim() < 2 || dual({&x, &gamma, &beta})) Py_RETURN_NONE;
    const auto dev = x.device();
    const int64_t D = x.size(-1), rows = x.numel() / (D ? D : 1);
    const bool graph = a[8] == Py_True && wants_grad({&x, &gamma, &beta});
    if (!ready(x, dev) || !ready(gamma, dev) || !ready(beta, dev) || D % 8 || D > (graph ? 2048 : 8192) || rows < 1 || gamma.numel() != D ||
        beta.numel() != D) Py_RETURN_NONE;
    const bool unpack = seq_offsets.defined();
    if (unpack && (!plain(seq_offsets, dev, at::kInt) || seq_offsets.numel() != B + 1 || !row_map.defined() || !plain(row_map, dev, at::kInt))) Py_RETURN_NONE;
    Tensor out;
    without_lock(x, [&] {
      out = unpack ? fresh(x, {B, L, D}) : fresh(x, x.sizes());
      norm(out, {x.const_data_ptr(), D}, {nullptr, 0}, gamma, beta, unpack ? B * L : rows, D, eps, seq_offsets, L);
      return true;
    });
    if (graph) {
      auto node = std::shared_ptr<FinalNormBackward>(new FinalNormBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(x, gamma, beta));
      node->x = keep(x);
      node->gamma = keep(gamma);
      node->beta = keep(beta);
      if ((node->packed = unpack)) node->row_map = keep(row_map);
      node->eps = eps;
      torch::autograd::set_history(out, node);
    }
    return THPVariable_Wrap(std::move(out));
  });
}

// linear(x [.., K], w [K, N], differentiable) -> x w, or None
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 3) {
    PyErr_SetString(PyExc_TypeError, "linear takes 3 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor x, w;
    if (!tensor_arg(a[0], &x) || !tensor_arg(a[1], &w) || !x.defined() || !w.defined() || !x.is_cuda() || x.dim() < 2 || w.dim() != 2 ||
        dual({&x, &w})) Py_RETURN_NONE;
    const auto dev = x.device();
    const int64_t K = w.size(0), N = w.size(1), M = x.numel() / (K ? K : 1);
    if (!ready(x, dev) || !ready(w, dev) || x.size(-1) != K || K % 8 || N % 8 || K < 8 || N < 8 || M < 1 || M > (1 << 30) || N > (1 << 30)) Py_RETURN_NONE;
    Tensor out;
    without_lock(x, [&] {
      auto shape = x.sizes().vec();
      shape.back() = N;
      out = fresh(x, shape);
      gemm(HSTU_GEMM_NN, M, {x.const_data_ptr(), K}, {&w}, K, N, out);
      return true;
    });
    if (a[2] == Py_True && wants_grad({&x, &w})) {
      auto node = std::shared_ptr<LinearBackward>(new LinearBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(x, w));
      node->x = keep(x);
      node->w = keep(w);
      torch::autograd::set_history(out, node);
    }
    return THPVariable_Wrap(std::move(out));
  });
}

// pack(lens, length) -> (seq_offsets, row_map, tokens) of the batch's packed form, or None.  Waits for the token count.
PyObject* pack(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 2) {
    PyErr_SetString(PyExc_TypeError, "pack takes 2 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor lens;
    int64_t L;
    if (!tensor_arg(a[0], &lens) || !lens.defined() || !long_arg(a[1], &L) || !lens.is_cuda() || lens.dim() != 1 || lens.size(0) < 1 || L < 1 ||
        !lens.is_contiguous() || (lens.scalar_type() != at::kInt && lens.scalar_type() != at::kLong) || lens.size(0) * L > 0x7fffffff) Py_RETURN_NONE;
    Tensor offsets, row_map;
    const int64_t T = without_lock(lens, [&]() -> int64_t {
      const int64_t B = lens.size(0);
      offsets = at::empty({B + 1}, lens.options().dtype(at::kInt).requires_grad(false));
      row_map = at::empty({B * L}, offsets.options());
      Word total(lens);
      void* const st = stream_of(lens);
      block_check(hstu_pack_plan(lens.const_data_ptr(), lens.scalar_type() == at::kLong, (int32_t)B, (int32_t)L, offsets.data_ptr<int32_t>(),
                                 row_map.data_ptr<int32_t>(), total.host.data_ptr<int32_t>(), st), "hstu_pack_plan");
      total.record(st);
      return total.wait();
    });
    return Py_BuildValue("(NNL)", THPVariable_Wrap(offsets), THPVariable_Wrap(row_map), (long long)T);
  });
}

// mask_lengths(mask [B, L] of bytes) -> (lengths int32 [B], ticket) or None; raised(ticket) -> whether a row was not end-padded.
// Two steps, so that the work on the lengths is enqueued before anyone waits.
PyObject* mask_lengths(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 1) {
    PyErr_SetString(PyExc_TypeError, "mask_lengths takes 1 argument");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Tensor mask;
    if (!tensor_arg(a[0], &mask) || !mask.defined() || !byte_mask(mask)) Py_RETURN_NONE;
    Tensor lens;
    auto word = without_lock(mask, [&] {
      lens = at::empty({mask.size(0)}, mask.options().dtype(at::kInt));
      auto bad = std::make_unique<Word>(mask);
      void* const st = stream_of(mask);
      block_check(hstu_mask_lengths((const uint8_t*)mask.const_data_ptr(), (int32_t)mask.size(0), (int32_t)mask.size(1), lens.data_ptr<int32_t>(),
                                    bad->host.data_ptr<int32_t>(), st), "hstu_mask_lengths");
      bad->record(st);
      return bad;
    });
    PyObject* const ticket = ticket_of(std::move(word));
    return ticket ? Py_BuildValue("(NN)", THPVariable_Wrap(lens), ticket) : nullptr;
  });
}

// has_room(device index, bytes): whether a buffer that a call can do without should be asked for.
PyObject* room(PyObject*, PyObject* const* a, Py_ssize_t count) {
  if (count != 2) {
    PyErr_SetString(PyExc_TypeError, "has_room takes 2 arguments");
    return nullptr;
  }
  const long device = PyLong_AsLong(a[0]);
  const long long bytes = PyLong_AsLongLong(a[1]);
  if (PyErr_Occurred()) return nullptr;
  return guarded([&]() -> PyObject* { return PyBool_FromLong(has_room((c10::DeviceIndex)device, (size_t)bytes)); });
}

PyMethodDef methods[] = {
    {"attention", (PyCFunction)(void (*)(void))attention, METH_FASTCALL,
     "One attention forward on arguments that are ready for the kernels; None when they are not."},
#define HSTU_FAST(name, doc) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, doc}
    HSTU_FAST(block, "One HSTU block forward (differentiable where asked)."),
    HSTU_FAST(blocks, "Several narrow HSTU blocks in inference as one launch."),
    HSTU_FAST(norm_gate_bwd, "The gradients of the norm and gate step."),
    HSTU_FAST(embed, "The model's front end: gather, position embedding, layer norm."),
    HSTU_FAST(final_norm, "The closing layer norm, into the padded batch where asked."),
    HSTU_FAST(linear, "A matrix product with gradients."),
    HSTU_FAST(pack, "The packed form of a padded batch."),
    HSTU_FAST(mask_lengths, "Lengths of an end-padded batch from its mask."),
    {"has_room", (PyCFunction)(void (*)(void))room, METH_FASTCALL, "Whether the device has room for a buffer that a call can do without."},
    {"raised", raised, METH_O, "Whether the kernel behind a ticket found what it looks for (waits for that kernel)."},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }

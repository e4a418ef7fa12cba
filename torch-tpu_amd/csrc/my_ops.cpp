// Operator registration of the MoE path, the way the reference does it: a C++ extension with
//     TORCH_LIBRARY(my_ops, m) { m.def("fused_moe_fused_experts", fused_moe_fused_experts); ... }
// (torch_tpu/csrc/ops/my_ops/myOps.cpp:29-80) - function pointers, schemas inferred, all arguments positional, caller
// allocated outputs, the output alias returned, argument errors through TORCH_CHECK (fusedMoE.cpp:143,148,231).
// Signatures follow torch_tpu/csrc/ops/my_ops/ops.hpp:610-676 and 716-722.
//
// The ops forward to the C ABI of libmoe_hip.so (include/moe_hip.h) on the current HIP stream.  Plain host C++
// against the torch headers; no device code here.  What the common call needs lives here: argument checks, the
// packed copy of the reference-layout weights (made once per weight set, found again through the identity of the
// sources' storages), one workspace per (device, stream).  The rarer forms of the op - bf16 weights, block sizes
// other than 128, ragged sizes, the W8A16 arithmetic - are handed to `my_ops::_fused_experts_general`, which the
// Python package defines on the same C ABI.  The dense ops mm_w8a16_dq_forward and mlp_w8a16_dq_forward are split the
// same way (`_mm_general`, `_mlp_general`): at decode sizes a call took longer in Python (21 us for the 7168 -> 1536 product
// at 32 rows, 7 us here) than its two launches take on the GPU (9 us).
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/library.h>

#include <algorithm>
#include <array>
#include <cstdio>
#include <map>
#include <memory>
#include <mutex>
#include <optional>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/moe_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

void check_rc(int rc, const char *what) { TORCH_CHECK(rc == 0, what, ": ", moe_hip_strerror(rc), " (code ", rc, ")"); }

c10::hip::HIPStream hip_stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()); }
void *stream_of(const Tensor &t) { return (void *)hip_stream_of(t).stream(); }

// ---- packed copies of weights -----------------------------------------------------------------------------------
// A packed copy belongs to the STORAGES of the tensors it was made from (not to the Python or C++ wrapper objects,
// which callers re-create freely: `param.data`, views made per call): storage, offset, shape, strides and dtype.  The entry
// keeps weak references to the storages; once one of them has been freed the entry is dead and is dropped by one of the next
// calls, and the storage's address is not given to another storage before that, so new weights never meet an old copy.  When the version counter of a
// source has moved the copy is made again, in the same memory: an update costs no memory, and a HIP graph that reads the
// copy goes on with the new weights (an update through the sources has to be ordered against their readers on other streams
// by whoever makes it, and the copy's readers are theirs).  An in-place write that does not move the version counter cannot
// be seen from here (my_ops::_invalidate_weight_cache after such an update).
// (two or three dimensions: the callers of identify() have checked that)
struct SourceId {
  const c10::StorageImpl *storage;
  const void *data;
  int64_t offset;
  c10::ScalarType dtype;
  int64_t sizes[3], strides[3];
  bool operator==(const SourceId &o) const {
    bool same = storage == o.storage && data == o.data && offset == o.offset && dtype == o.dtype;
    for (int i = 0; i < 3; i++) same = same && sizes[i] == o.sizes[i] && strides[i] == o.strides[i];
    return same;
  }
};

SourceId identify(const Tensor &t) {
  SourceId s{};
  s.storage = t.unsafeGetTensorImpl()->unsafe_storage().unsafeGetStorageImpl();
  s.data = t.data_ptr();
  s.offset = t.storage_offset();
  s.dtype = t.scalar_type();
  for (int i = 0; i < 3 && i < t.dim(); i++) {
    s.sizes[i] = t.size(i);
    s.strides[i] = t.stride(i);
  }
  return s;
}

uint32_t version_of(const Tensor &t) { return t.is_inference() ? 0u : (uint32_t)t._version(); }

enum PackedForm { kFormExperts, kFormMm, kFormMlp };
constexpr int kMaxSources = 6, kMaxMade = 4;

// An event behind the work that makes a copy, until that work has been seen complete
struct ReadyEvent {
  hipEvent_t event = nullptr;
  ReadyEvent() = default;
  ReadyEvent(ReadyEvent &&o) noexcept : event(o.event) { o.event = nullptr; }
  ReadyEvent &operator=(ReadyEvent &&) = delete;
  ~ReadyEvent() { drop(); }
  void drop() {
    if (event) (void)hipEventDestroy(event);
    event = nullptr;
  }
  void record(hipStream_t st) {
    if (!event) C10_HIP_CHECK(hipEventCreateWithFlags(&event, hipEventDisableTiming));
    C10_HIP_CHECK(hipEventRecord(event, st));
  }
  // whether the work is known to be complete (asked in a way that a capture, this thread's or another's, allows)
  bool complete() {
    if (!event) return true;
    c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
    const hipError_t rc = hipEventQuery(event);
    if (rc == hipSuccess) {
      drop();
      return true;
    }
    (void)hipGetLastError();
    if (rc != hipErrorNotReady) C10_HIP_CHECK(rc);
    return false;
  }
};

struct PackedEntry {
  PackedForm form;
  std::array<SourceId, kMaxSources> ids{};
  std::array<uint32_t, kMaxSources> versions{};
  std::vector<c10::weak_intrusive_ptr<c10::StorageImpl>> alive;
  std::array<Tensor, kMaxMade> made;      // tile-blocked weights and fp32 scales, one pair (a product) or two
  ReadyEvent ready;                       // behind the launches that filled `made`
  std::vector<c10::hip::HIPStream> known_to_allocator;    // streams whose work the copies' memory waits for when it is freed
  int64_t packings = 0;
  int64_t rows = 0;                       // dense: the largest batch seen and the workspace that covers it and all smaller ones
  size_t workspace_bytes = 0;
  bool dead() const {
    for (auto &w : alive)
      if (w.expired()) return true;
    return false;
  }
};

std::mutex g_mutex;
// The entries, and a hash of each one's form and sources beside them: a call compares hashes, one cache line for eight
// entries, and looks closer at a match.  (Reading every entry and its weak references instead: 8.5 us a call against 8.3 with 610
// weights, 8.2 against 8.1 with 305.)
struct PackedTable {
  std::vector<std::unique_ptr<PackedEntry>> entries;
  std::vector<size_t> hashes;
  size_t next_look = 0;

  static size_t hash_of(PackedForm form, const std::array<SourceId, kMaxSources> &ids) {
    size_t h = form;
    for (const SourceId &s : ids) h = (h ^ (size_t)s.data ^ ((size_t)s.storage >> 4)) * 0x9e3779b97f4a7c15ull + (size_t)s.sizes[0];
    return h;
  }
  PackedEntry *find(PackedForm form, const std::array<SourceId, kMaxSources> &ids, size_t hash) {
    for (size_t i = 0; i < hashes.size(); i++)
      if (hashes[i] == hash && entries[i]->form == form && entries[i]->ids == ids) return entries[i].get();
    return nullptr;
  }
  PackedEntry *add(size_t hash) {
    entries.push_back(std::make_unique<PackedEntry>());
    hashes.push_back(hash);
    return entries.back().get();
  }
  void drop(size_t i) {
    entries[i] = std::move(entries.back());
    entries.pop_back();
    hashes[i] = hashes.back();
    hashes.pop_back();
  }
  void drop(const PackedEntry *e) {
    for (size_t i = 0; i < entries.size(); i++)
      if (entries[i].get() == e) return drop(i);
  }
  // every call looks at a few entries in turn for dead ones, one that packs at all of them
  void drop_dead(size_t looks) {
    for (; looks && !entries.empty(); looks--) {
      if (next_look >= entries.size()) next_look = 0;
      if (entries[next_look]->dead()) drop(next_look);
      else next_look++;
    }
  }
  void drop_all_dead() { drop_dead(entries.size()); }
};
PackedTable &g_packed = *new PackedTable;      // (no events destroyed after the runtime at exit)
std::map<std::pair<int, void *>, Tensor> g_workspace, g_rw;
int g_numerics = 0;     // 0 = w8a8 (this file), 1 = w8a16 (general path)

// row-major weight bytes -> tile-blocked (moe_pack_weights), into the copy that is there or a new one
void put_weights(Tensor &dst, const Tensor &rowmajor) {
  const Tensor w = rowmajor.contiguous();
  if (!dst.defined()) dst = at::empty_like(w);
  check_rc(moe_pack_weights(stream_of(w), w.data_ptr(), w.numel() / w.size(-1), (int)(w.size(-1) * w.element_size()),
                            dst.data_ptr()),
           "moe_pack_weights");
}

// Block scales as fp32, contiguous, in memory of their own: `to` and `contiguous` hand an fp32 tensor through as it is, and
// an entry that holds its source's storage never sees it die
void put_scales(Tensor &dst, const Tensor &s) {
  if (!dst.defined()) dst = at::empty(s.sizes(), s.options().dtype(at::kFloat));
  dst.copy_(s);
}

// Packed copies are plain data: made outside autograd (a recorded cat or cast would hold the source parameter) and as normal
// tensors also inside inference mode
struct PackGuard {
  c10::InferenceMode inference{false};
  at::NoGradGuard no_grad;
};

// What a call multiplies with: an entry's copies, or some of its own
struct Packed {
  std::array<Tensor, kMaxMade> made;
  PackedEntry *entry;           // null: a copy that lives in a captured graph
};

// Call with g_mutex held; make(made) fills or refills the copies.  The copies are made on the caller's stream; a call on
// another stream waits for that on its own stream, without holding up the host, and the allocator is told of it once.  Work
// under capture runs with every replay and not now, so nothing that it makes is left for other calls to find: a weight set
// that has no finished copy then (warm up first) is packed inside the graph.
template <typename Make>
Packed packed(PackedForm form, std::initializer_list<const Tensor *> src, Make make) {
  std::array<SourceId, kMaxSources> ids{};
  std::array<uint32_t, kMaxSources> versions{};
  int n = 0;
  for (const Tensor *t : src) {
    ids[n] = identify(*t);
    versions[n++] = version_of(*t);
  }
  const c10::hip::HIPStream stream = hip_stream_of(**src.begin());
  const auto capturing = [&] {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    C10_HIP_CHECK(hipStreamIsCapturing(stream.stream(), &status));
    return status != hipStreamCaptureStatusNone;
  };
  const size_t hash = PackedTable::hash_of(form, ids);
  g_packed.drop_dead(4);
  PackedEntry *found = g_packed.find(form, ids, hash);
  const bool current = found && found->versions == versions;
  if (!(current && found->ready.complete()) && capturing()) {
    PackGuard guard;
    Packed own{{}, nullptr};
    make(own.made);
    return own;
  }
  if (!found) {
    g_packed.drop_all_dead();
    found = g_packed.add(hash);
    found->form = form;
    found->ids = ids;
    for (const Tensor *t : src) found->alive.push_back(t->storage().getWeakStorageImpl());
    found->known_to_allocator.push_back(stream);
  } else if (found->ready.event) {
    C10_HIP_CHECK(hipStreamWaitEvent(stream.stream(), found->ready.event, 0));
  }
  if (!current) {
    try {
      PackGuard guard;
      c10::DeviceGuard device((*src.begin())->device());
      make(found->made);
      found->ready.record(stream.stream());
    } catch (...) {
      g_packed.drop(found);
      throw;
    }
    found->versions = versions;
    found->packings++;
  }
  auto &known = found->known_to_allocator;
  if (std::find(known.begin(), known.end(), stream) == known.end()) {
    for (const Tensor &t : found->made)
      if (t.defined()) c10::hip::HIPCachingAllocator::recordStream(t.storage().data_ptr(), stream);
    known.push_back(stream);
  }
  return {found->made, found};
}

// Reference argument layout (gate [E,I,H], up [E,I,H], down pre-transposed [E,I,H], bf16 scales of the same
// orientation: python/regression/test_llm/test_moe.py:285-288) -> W13 = gate rows then up rows [E,2I,H], its scales, W2 =
// down in checkpoint orientation [E,H,I], its scales; scales widened to fp32, weight bytes tile-blocked.  Values are
// untouched.  The gated MLP's weights are the same without the expert dimension.
Packed packed_gated(PackedForm form, const Tensor &gate, const Tensor &up, const Tensor &down, const Tensor &gs,
                    const Tensor &us, const Tensor &ds) {
  return packed(form, {&gate, &up, &down, &gs, &us, &ds}, [&](std::array<Tensor, kMaxMade> &made) {
    put_weights(made[0], at::cat({gate, up}, -2));
    put_scales(made[1], at::cat({gs, us}, -2));
    put_weights(made[2], down.transpose(-2, -1));
    put_scales(made[3], ds.transpose(-2, -1));
  });
}

Packed packed_mm(const Tensor &weight, const Tensor &scale) {
  return packed(kFormMm, {&weight, &scale}, [&](std::array<Tensor, kMaxMade> &made) {
    put_weights(made[0], weight);
    put_scales(made[1], scale);
  });
}

// Workspace of a call on M rows: asked for again only when a batch is larger than every one before it (the query looks at
// all smaller batches), so that a layer's later, smaller calls never grow the scratch
template <typename Query>
size_t dense_workspace(PackedEntry *e, int64_t M, Query query) {
  if (!e) return query();
  if (M > e->rows) {
    e->workspace_bytes = query();
    e->rows = M;
  }
  return e->workspace_bytes;
}

// what the common forms of the dense ops ask of their tensors; any other form takes the general road
bool plain_matrix(const Tensor &t, c10::ScalarType dtype, int64_t rows, int64_t cols, const Tensor &like) {
  return t.dim() == 2 && t.scalar_type() == dtype && t.size(0) == rows && t.size(1) == cols && t.is_cuda() &&
         t.device() == like.device() && t.is_contiguous() && (uintptr_t)t.const_data_ptr() % 16 == 0;
}
bool plain_weight(const Tensor &w, const Tensor &s, int64_t rows, int64_t cols, const Tensor &like) {
  return w.dim() == 2 && w.scalar_type() == at::kFloat8_e4m3fn && w.size(0) == rows && w.size(1) == cols && w.is_cuda() &&
         w.device() == like.device() && !w.is_inference() && s.dim() == 2 && s.size(0) == (rows + 127) / 128 &&
         s.size(1) == (cols + 127) / 128 && s.is_cuda() && s.device() == like.device() && !s.is_inference();
}

// one scratch tensor per (device, stream), grown on demand: nothing is allocated once it is large enough
Tensor &scratch(std::map<std::pair<int, void *>, Tensor> &table, const Tensor &like, void *stream, size_t bytes,
                size_t floor_bytes) {
  Tensor &t = table[{(int)like.device().index(), stream}];
  if (!t.defined() || (size_t)t.numel() < bytes)
    t = at::empty({(int64_t)std::max(bytes, floor_bytes)}, like.options().dtype(at::kByte));
  return t;
}

// ---- enable_profile / disable_profile (torch_tpu/csrc/ops/my_ops/profile.cpp:12-44) --------------------------------
// While enabled, the expert and routing ops of this file bracket their work on the stream with a pair of events; disable_profile waits
// for them and reports GPU time per op (count, total, mean, min, max).  At most `max_record_num` calls are recorded.
struct ProfileRecord {
  const char *op;
  hipEvent_t start, stop;
};
bool g_profiling = false;
int64_t g_profile_max = 0, g_profile_mode = 0;
std::vector<ProfileRecord> g_profile;
std::string g_profile_report;

struct ProfileScope {
  hipEvent_t stop = nullptr;
  void *stream = nullptr;
  // call with g_mutex held
  ProfileScope(const char *op, void *st) {
    if (!g_profiling || (int64_t)g_profile.size() >= g_profile_max) return;
    ProfileRecord r{op, nullptr, nullptr};
    if (hipEventCreate(&r.start) != hipSuccess) return;
    if (hipEventCreate(&r.stop) != hipSuccess) {
      (void)hipEventDestroy(r.start);
      return;
    }
    (void)hipEventRecord(r.start, (hipStream_t)st);
    stop = r.stop;
    stream = st;
    g_profile.push_back(r);
  }
  ~ProfileScope() {
    if (stop) (void)hipEventRecord(stop, (hipStream_t)stream);
  }
};

Tensor call_general(const char *name, std::vector<c10::IValue> stack) {
  auto op = c10::Dispatcher::singleton().findSchema({name, ""});
  TORCH_CHECK(op.has_value(), name, " is not defined: this form of the op is implemented by the Python package "
              "(import torch_tpu_amd)");
  op->callBoxed(stack);
  return stack.at(0).toTensor();
}

}  // namespace

namespace at {

Tensor fused_moe_fused_experts(const Tensor &output, const Tensor &input, const OptTensor &output_sample,
                               const OptTensor &input_sample, const Tensor &gate_weights, const Tensor &up_weights,
                               const Tensor &down_weights, const OptTensor &gate_scales, const OptTensor &up_scales,
                               const OptTensor &down_scales, const Tensor &select_experts, const Tensor &routing_weights,
                               const OptTensor &num_select_experts, const OptTensor &select_experts_middle,
                               const OptTensor &routing_weights_middle, int64_t blocksize, int64_t num_experts,
                               int64_t num_experts_per_tok, bool use_grouped_topk, int64_t num_expert_group,
                               int64_t topk_group, const OptTensor &silu, const OptTensor &sigmoid, const OptTensor &m0,
                               bool save_mid_res) {
  TORCH_CHECK(select_experts.scalar_type() == at::kInt, "select_experts must be int32 dtype");
  if (num_select_experts.has_value())
    TORCH_CHECK(num_select_experts->scalar_type() == at::kLong, "num_select_experts must be int64 dtype");
  const std::pair<const char *, const OptTensor *> unpinned[] = {
      {"output_sample", &output_sample}, {"input_sample", &input_sample}, {"num_select_experts", &num_select_experts},
      {"silu", &silu},                   {"sigmoid", &sigmoid},           {"m0", &m0}};
  for (auto &p : unpinned)
    TORCH_CHECK(!p.second->has_value(), p.first, ": the reference never passes this argument and leaves its meaning "
                "undefined; it is not supported");
  TORCH_CHECK(!save_mid_res, "save_mid_res is not supported");

  const bool scaled = gate_scales.has_value() && up_scales.has_value() && down_scales.has_value();
  bool fast = scaled && blocksize == 128 && g_numerics == 0 && input.dim() == 2 && gate_weights.dim() == 3 &&
              select_experts.dim() == 2 && (output.dim() == 2 || output.dim() == 3);
  if (fast) {
    const int64_t I = gate_weights.size(1), H = gate_weights.size(2);
    fast = I % 128 == 0 && H % 128 == 0 && input.size(1) == H && gate_weights.scalar_type() == at::kFloat8_e4m3fn &&
           up_weights.scalar_type() == at::kFloat8_e4m3fn && down_weights.scalar_type() == at::kFloat8_e4m3fn &&
           up_weights.sizes() == gate_weights.sizes() && down_weights.sizes() == gate_weights.sizes() &&
           gate_scales->dim() == 3 && gate_scales->sizes() == up_scales->sizes() &&
           gate_scales->sizes() == down_scales->sizes() && gate_scales->size(1) == I / 128 &&
           gate_scales->size(2) == H / 128;
  }
  if (!fast) {
    return call_general("my_ops::_fused_experts_general",
                        {output, input, output_sample, input_sample, gate_weights, up_weights, down_weights, gate_scales,
                         up_scales, down_scales, select_experts, routing_weights, num_select_experts, select_experts_middle,
                         routing_weights_middle, blocksize, num_experts, num_experts_per_tok, use_grouped_topk,
                         num_expert_group, topk_group, silu, sigmoid, m0, save_mid_res});
  }

  const int64_t T = input.size(0), H = input.size(1), E = gate_weights.size(0), I = gate_weights.size(1);
  const int64_t K = select_experts.size(1);
  TORCH_CHECK(E == num_experts && K == num_experts_per_tok, "num_experts / num_experts_per_tok do not match the tensors");
  for (const Tensor *t : {&output, &input, &gate_weights, &up_weights, &down_weights, &*gate_scales, &*up_scales,
                          &*down_scales, &select_experts})
    TORCH_CHECK(t->is_cuda() && t->is_contiguous(), "tensors must be contiguous and on the GPU");
  TORCH_CHECK(input.scalar_type() == at::kBFloat16 && output.scalar_type() == at::kBFloat16,
              "input and output must be bfloat16");
  TORCH_CHECK(select_experts.size(0) == T, "select_experts must be [T, K]");
  const int out_mode = output.dim() == 2 ? 1 : 0;
  if (out_mode) {
    TORCH_CHECK(output.size(0) == T && output.size(1) == H, "output must be [T,H] or [T,K,H]");
  } else {
    TORCH_CHECK(output.size(0) == T && output.size(1) == K && output.size(2) == H, "output must be [T,H] or [T,K,H]");
  }

  std::lock_guard<std::mutex> lock(g_mutex);
  void *st = stream_of(input);
  ProfileScope prof("fused_moe_fused_experts", st);
  const auto w = packed_gated(kFormExperts, gate_weights, up_weights, down_weights, *gate_scales, *up_scales, *down_scales).made;
  const void *rw = nullptr;
  int rw_dtype = MOE_DTYPE_F32;
  if (out_mode) {
    // [T,H] form: the fp32 weighted sum over the slots; the reference's callers hold the weights in bf16, which the
    // library widens inside the sum
    TORCH_CHECK(routing_weights.dim() == 2 && routing_weights.size(0) == T && routing_weights.size(1) == K &&
                routing_weights.is_cuda(), "routing_weights must be [T, K]");
    if (routing_weights.scalar_type() == at::kFloat && routing_weights.is_contiguous()) {
      rw = routing_weights.data_ptr();
    } else if (routing_weights.scalar_type() == at::kBFloat16 && routing_weights.is_contiguous()) {
      rw = routing_weights.data_ptr();
      rw_dtype = MOE_DTYPE_BF16;
    } else {
      Tensor &buf = scratch(g_rw, input, st, (size_t)(T * K) * 4, 16384);
      Tensor view = buf.narrow(0, 0, T * K * 4).view(at::kFloat).view({T, K});
      view.copy_(routing_weights);
      rw = view.data_ptr();
    }
  }
  const size_t need = moe_fused_experts_workspace_bytes((int)T, (int)H, (int)I, (int)E, (int)K, 0);
  Tensor &ws = scratch(g_workspace, input, st, need, (size_t)1 << 20);
  check_rc(moe_fused_experts_fp8_rw(st, input.data_ptr(), (int)T, (int)H, (const uint8_t *)w[0].data_ptr(),
                                    w[1].data_ptr<float>(), (const uint8_t *)w[2].data_ptr(), w[3].data_ptr<float>(),
                                    (int)I, (int)E, select_experts.data_ptr<int32_t>(), rw, rw_dtype, (int)K, nullptr,
                                    nullptr, nullptr, nullptr, 0, output.data_ptr(), out_mode, ws.data_ptr(),
                                    (size_t)ws.numel()),
           "fused_moe_fused_experts");
  return output;
}

// the second implementation of the reference (fusedMoE.cpp:237-318): same result; its scratch tensors are accepted
// and left untouched
Tensor fused_moe_fused_experts_v2(const Tensor &output, const Tensor &input, const OptTensor &output_sample,
                                  const OptTensor &input_sample, const Tensor &gate_weights, const Tensor &up_weights,
                                  const Tensor &down_weights, const OptTensor &gate_scales, const OptTensor &up_scales,
                                  const OptTensor &down_scales, const Tensor &select_experts,
                                  const Tensor &routing_weights, const OptTensor &num_select_experts,
                                  const OptTensor &select_experts_middle, const OptTensor &routing_weights_middle,
                                  const OptTensor &gather_buffer, const OptTensor &scatter_buffer, int64_t blocksize,
                                  int64_t num_experts, int64_t num_experts_per_tok, bool use_grouped_topk,
                                  int64_t num_expert_group, int64_t topk_group, const OptTensor &silu,
                                  const OptTensor &sigmoid, const OptTensor &m0, bool save_mid_res) {
  return fused_moe_fused_experts(output, input, output_sample, input_sample, gate_weights, up_weights, down_weights,
                                 gate_scales, up_scales, down_scales, select_experts, routing_weights, num_select_experts,
                                 select_experts_middle, routing_weights_middle, blocksize, num_experts,
                                 num_experts_per_tok, use_grouped_topk, num_expert_group, topk_group, silu, sigmoid, m0,
                                 save_mid_res);
}

// torch_tpu/csrc/ops/my_ops/MmW8A16Dq.cpp:185-228: weight [N, K], scale [ceil(N/bs), ceil(K/bs)], output [M, N]
Tensor mm_w8a16_dq_forward(const Tensor &input, const Tensor &weight, const Tensor &scale, const Tensor &output,
                           int64_t blocksize) {
  bool fast = blocksize == 128 && input.dim() == 2 && weight.dim() == 2;
  const int64_t M = fast ? input.size(0) : 0, N = fast ? weight.size(0) : 0, K = fast ? weight.size(1) : 0;
  fast = fast && M > 0 && K >= 128 && K % 128 == 0 && K <= 32768 && N >= 16 && N % 16 == 0 && N <= (1 << 20) &&
         M * K < (1ll << 31) && M * N < (1ll << 31) && N * K < (1ll << 32) && plain_weight(weight, scale, N, K, input) &&
         plain_matrix(input, at::kBFloat16, M, K, input) && plain_matrix(output, at::kBFloat16, M, N, input);
  std::unique_lock<std::mutex> lock(g_mutex);
  if (!fast || g_numerics != 0) {
    lock.unlock();
    return call_general("my_ops::_mm_general", {input, weight, scale, output, blocksize});
  }
  void *st = stream_of(input);
  const Packed p = packed_mm(weight, scale);
  const auto &w = p.made;
  const size_t need = dense_workspace(p.entry, M, [&] { return moe_mm_fp8_workspace_bytes((int)M, (int)K, (int)N); });
  Tensor &ws = scratch(g_workspace, input, st, need, (size_t)1 << 20);
  check_rc(moe_mm_fp8(st, input.data_ptr(), (int)M, (int)K, (const uint8_t *)w[0].data_ptr(), w[1].data_ptr<float>(), (int)N,
                      output.data_ptr(), ws.data_ptr(), (size_t)ws.numel()),
           "mm_w8a16_dq_forward");
  return output;
}

// torch_tpu/csrc/ops/my_ops/MlpW8A16Dq.cpp:189-241: gate / up [I, H], down passed transposed as [I, H], scales likewise
Tensor mlp_w8a16_dq_forward(const Tensor &input, const Tensor &gate, const Tensor &up, const Tensor &down, const Tensor &gs,
                            const Tensor &us, const Tensor &ds, const Tensor &output, int64_t blocksize) {
  bool fast = blocksize == 128 && input.dim() == 2 && gate.dim() == 2;
  const int64_t M = fast ? input.size(0) : 0, I = fast ? gate.size(0) : 0, H = fast ? gate.size(1) : 0;
  fast = fast && M > 0 && H >= 128 && H % 128 == 0 && H <= 32768 && I >= 128 && I % 128 == 0 && I <= 32768 &&
         M * H < (1ll << 31) && M * I < (1ll << 31) && plain_weight(gate, gs, I, H, input) &&
         plain_weight(up, us, I, H, input) && plain_weight(down, ds, I, H, input) && gs.scalar_type() == us.scalar_type() &&
         plain_matrix(input, at::kBFloat16, M, H, input) && plain_matrix(output, at::kBFloat16, M, H, input);
  std::unique_lock<std::mutex> lock(g_mutex);
  if (!fast || g_numerics != 0) {
    lock.unlock();
    return call_general("my_ops::_mlp_general", {input, gate, up, down, gs, us, ds, output, blocksize});
  }
  void *st = stream_of(input);
  const Packed p = packed_gated(kFormMlp, gate, up, down, gs, us, ds);
  const auto &w = p.made;
  const size_t need = dense_workspace(p.entry, M, [&] { return moe_mlp_fp8_workspace_bytes((int)M, (int)H, (int)I); });
  Tensor &ws = scratch(g_workspace, input, st, need, (size_t)1 << 20);
  check_rc(moe_mlp_fp8(st, input.data_ptr(), (int)M, (int)H, (const uint8_t *)w[0].data_ptr(), w[1].data_ptr<float>(),
                       (const uint8_t *)w[2].data_ptr(), w[3].data_ptr<float>(), (int)I, output.data_ptr(), ws.data_ptr(),
                       (size_t)ws.numel()),
           "mlp_w8a16_dq_forward");
  return output;
}

// The packed copies for the other roads of the dense ops (strided tensors, the W8A16 arithmetic, mlp_w8a8_quant_forward):
// a weight is packed once, whatever form its calls take.  Empty: not the form of weights that this file packs.
std::vector<Tensor> _mm_weights(const Tensor &weight, const Tensor &scale) {
  if (weight.dim() != 2 || weight.size(0) % 16 || weight.size(1) % 128 ||
      !plain_weight(weight, scale, weight.size(0), weight.size(1), weight))
    return {};
  std::lock_guard<std::mutex> lock(g_mutex);
  const Packed p = packed_mm(weight, scale);
  return {p.made[0].detach(), p.made[1].detach()};
}

std::vector<Tensor> _mlp_weights(const Tensor &gate, const Tensor &up, const Tensor &down, const Tensor &gs, const Tensor &us,
                                 const Tensor &ds) {
  if (gate.dim() != 2) return {};
  const int64_t I = gate.size(0), H = gate.size(1);
  if (I % 128 || H % 128 || !plain_weight(gate, gs, I, H, gate) || !plain_weight(up, us, I, H, gate) ||
      !plain_weight(down, ds, I, H, gate) || gs.scalar_type() != us.scalar_type())
    return {};
  std::lock_guard<std::mutex> lock(g_mutex);
  const Packed p = packed_gated(kFormMlp, gate, up, down, gs, us, ds);
  return {p.made[0].detach(), p.made[1].detach(), p.made[2].detach(), p.made[3].detach()};
}

// torch_tpu/csrc/ops/my_ops/NoauxTcTopk.cpp:9-67: group-limited top-k into caller-allocated values / indices
Tensor noaux_tc_topk(const Tensor &values, const Tensor &indices, const Tensor &scores, int64_t n_groups,
                     int64_t topk_groups, int64_t top_k) {
  TORCH_CHECK(scores.dim() == 2, "scores must be 2D tensor");
  TORCH_CHECK(values.scalar_type() == scores.scalar_type(), "values and scores must have the same dtype");
  TORCH_CHECK(indices.scalar_type() == at::kInt, "indices must be int32");
  const int64_t T = scores.size(0), E = scores.size(1);
  TORCH_CHECK(values.dim() == 2 && values.size(0) == T && values.size(1) == top_k, "values shape must be [batch_size, top_k]");
  TORCH_CHECK(indices.dim() == 2 && indices.size(0) == T && indices.size(1) == top_k,
              "indices shape must be [batch_size, top_k]");
  TORCH_CHECK(n_groups > 0 && E % n_groups == 0, "total_size must be divisible by n_groups");
  TORCH_CHECK(topk_groups <= n_groups, "topk_groups must be <= n_groups");
  TORCH_CHECK(top_k > 0, "top_k must be positive");
  TORCH_CHECK(scores.scalar_type() == at::kFloat || scores.scalar_type() == at::kBFloat16,
              "scores must be float32 or bfloat16");
  for (const Tensor *t : {&values, &indices, &scores})
    TORCH_CHECK(t->is_cuda() && t->is_contiguous(), "tensors must be contiguous and on the GPU");
  std::lock_guard<std::mutex> lock(g_mutex);
  ProfileScope prof("noaux_tc_topk", stream_of(scores));
  check_rc(moe_noaux_tc_topk(stream_of(scores), scores.data_ptr(),
                             scores.scalar_type() == at::kFloat ? MOE_DTYPE_F32 : MOE_DTYPE_BF16, (int)T, (int)E,
                             (int)n_groups, (int)topk_groups, (int)top_k, values.data_ptr(), indices.data_ptr<int32_t>()),
           "noaux_tc_topk");
  return values;
}

// torch_tpu/csrc/ops/my_ops/fusedMoE.cpp:82-115: closed, untested and undocumented in the reference
Tensor fused_moe_grouped_topk(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                              const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &) {
  TORCH_CHECK(false, "fused_moe_grouped_topk: the reference's fused router is closed-source, untested and undocumented; "
              "use noaux_tc_topk or torch_tpu_amd.moe_route instead");
}

void enable_profile(std::optional<int64_t> max_record_num, std::optional<int64_t> mode) {
  std::lock_guard<std::mutex> lock(g_mutex);
  for (auto &r : g_profile) {
    (void)hipEventDestroy(r.start);
    (void)hipEventDestroy(r.stop);
  }
  g_profile.clear();
  g_profile_max = max_record_num.value_or(40960);          // the reference's defaults (profile.cpp:17-18)
  g_profile_mode = mode.value_or(1);
  TORCH_CHECK(g_profile_max >= 0, "max_record_num must not be negative");
  g_profiling = true;
}

void disable_profile() {
  std::lock_guard<std::mutex> lock(g_mutex);
  g_profiling = false;
  struct Sum {
    int64_t n = 0;
    double total = 0, lo = 1e300, hi = 0;
  };
  std::map<std::string, Sum> per_op;
  for (auto &r : g_profile) {
    float ms = 0.f;
    if (hipEventSynchronize(r.stop) == hipSuccess && hipEventElapsedTime(&ms, r.start, r.stop) == hipSuccess) {
      Sum &s = per_op[r.op];
      s.n++;
      s.total += ms * 1e3;
      s.lo = std::min(s.lo, (double)ms * 1e3);
      s.hi = std::max(s.hi, (double)ms * 1e3);
    }
    (void)hipEventDestroy(r.start);
    (void)hipEventDestroy(r.stop);
  }
  g_profile.clear();
  std::ostringstream os;
  os << "my_ops profile: op, calls, total us, mean us, min us, max us\n";
  for (auto &kv : per_op)
    os << kv.first << ", " << kv.second.n << ", " << kv.second.total << ", " << kv.second.total / kv.second.n << ", "
       << kv.second.lo << ", " << kv.second.hi << "\n";
  g_profile_report = os.str();
  if (g_profile_mode != 0) std::fputs(g_profile_report.c_str(), stdout);
}

std::string _profile_report() {
  std::lock_guard<std::mutex> lock(g_mutex);
  return g_profile_report;
}

// housekeeping for the Python package: the arithmetic switch and the packed-copy table
void _set_expert_numerics(int64_t mode) {
  TORCH_CHECK(mode == 0 || mode == 1, "mode must be 0 (w8a8) or 1 (w8a16)");
  std::lock_guard<std::mutex> lock(g_mutex);
  g_numerics = (int)mode;
}

void _invalidate_weight_cache() {
  std::lock_guard<std::mutex> lock(g_mutex);
  g_packed.entries.clear();
  g_packed.hashes.clear();
}

// weight sets packed for tensors that are alive, every update of one counted again
int64_t _packed_weight_sets() {
  std::lock_guard<std::mutex> lock(g_mutex);
  int64_t n = 0;
  g_packed.drop_all_dead();
  for (auto &e : g_packed.entries) n += e->packings;
  return n;
}

// ---- the layer's one call ---------------------------------------------------------------------------------------------
// moe_layer_fp8 for the common form of ops.layer_fp8: every operand plain and on the current device.  The checks and the call
// took 20 us of Python per layer call, as long as all launches of a small layer (256 x 512, 8 experts, 1 to 100 tokens).
// Returns the library's code, or kNotPlain for any other form: the caller's own road then says what is wrong, or runs it.
constexpr int64_t kNotPlain = 1 << 20;

bool plain_tensor(const Tensor &t, c10::ScalarType dtype, at::IntArrayRef sizes, const Tensor &like) {
  return t.scalar_type() == dtype && t.sizes() == sizes && t.is_cuda() && t.device() == like.device() && t.is_contiguous();
}

int64_t _layer_fp8(const Tensor &x, const Tensor &router, const Tensor &w13, const Tensor &w13s, const Tensor &w2, const Tensor &w2s,
                   int64_t top_k, int64_t mode, const OptTensor &bias, int64_t n_groups, int64_t topk_groups, bool renorm,
                   double scale, const OptTensor &sh13, const OptTensor &sh13s, const OptTensor &sh2, const OptTensor &sh2s,
                   const Tensor &out, const Tensor &workspace) {
  if (x.dim() != 2 || w13.dim() != 3 || !x.is_cuda() || x.device().index() != c10::hip::current_device()) return kNotPlain;
  const int64_t T = x.size(0), H = x.size(1), E = w13.size(0), I = w13.size(1) / 2;
  const auto fits = [](int64_t v) { return v >= 0 && v < (1ll << 31); };
  if (!fits(T) || !fits(H) || !fits(I) || E < 1 || E > 1024 || top_k < 1 || top_k > E || H % 128 || I % 128 || !fits(n_groups) ||
      !fits(topk_groups))
    return kNotPlain;
  const auto fp8 = at::kFloat8_e4m3fn;
  if (!plain_tensor(x, at::kBFloat16, {T, H}, x) || !plain_tensor(router, at::kBFloat16, {E, H}, x) ||
      !plain_tensor(w13, fp8, {E, 2 * I, H}, x) || !plain_tensor(w13s, at::kFloat, {E, 2 * I / 128, H / 128}, x) ||
      !plain_tensor(w2, fp8, {E, H, I}, x) || !plain_tensor(w2s, at::kFloat, {E, H / 128, I / 128}, x) ||
      !plain_tensor(out, at::kBFloat16, {T, H}, x) || !plain_tensor(workspace, at::kByte, {workspace.numel()}, x) ||
      (bias && !plain_tensor(*bias, at::kFloat, {E}, x)))
    return kNotPlain;
  int64_t I_sh = 0;
  if (sh13) {
    if (!sh13s || !sh2 || !sh2s || sh13->dim() != 3) return kNotPlain;
    I_sh = sh13->size(1) / 2;
    if (I_sh < 128 || I_sh % 128 || !fits(I_sh) || !plain_tensor(*sh13, fp8, {1, 2 * I_sh, H}, x) ||
        !plain_tensor(*sh13s, at::kFloat, {1, 2 * I_sh / 128, H / 128}, x) || !plain_tensor(*sh2, fp8, {1, H, I_sh}, x) ||
        !plain_tensor(*sh2s, at::kFloat, {1, H / 128, I_sh / 128}, x))
      return kNotPlain;
  }
  if ((size_t)workspace.numel() < moe_layer_fp8_workspace_bytes((int)T, (int)H, (int)I, (int)E, (int)top_k, (int)I_sh)) return kNotPlain;
  return moe_layer_fp8(stream_of(x), x.data_ptr(), (int)T, (int)H, router.data_ptr(), bias ? bias->data_ptr<float>() : nullptr,
                       (int)E, (int)top_k, (int)mode, (int)n_groups, (int)topk_groups, renorm, (float)scale,
                       (const uint8_t *)w13.data_ptr(), w13s.data_ptr<float>(), (const uint8_t *)w2.data_ptr(),
                       w2s.data_ptr<float>(), (int)I, sh13 ? (const uint8_t *)sh13->data_ptr() : nullptr,
                       sh13 ? sh13s->data_ptr<float>() : nullptr, sh13 ? (const uint8_t *)sh2->data_ptr() : nullptr,
                       sh13 ? sh2s->data_ptr<float>() : nullptr, (int)I_sh, out.data_ptr(), nullptr, nullptr, nullptr,
                       workspace.data_ptr(), (size_t)workspace.numel());
}

// memory that the packed copies hold
int64_t _packed_weight_bytes() {
  std::lock_guard<std::mutex> lock(g_mutex);
  int64_t n = 0;
  g_packed.drop_all_dead();
  for (auto &e : g_packed.entries)
    for (auto &t : e->made)
      if (t.defined()) n += (int64_t)t.nbytes();
  return n;
}

TORCH_LIBRARY(my_ops, m) {
  m.def("fused_moe_grouped_topk", fused_moe_grouped_topk);
  m.def("fused_moe_fused_experts", fused_moe_fused_experts);
  m.def("fused_moe_fused_experts_v2", fused_moe_fused_experts_v2);
  m.def("noaux_tc_topk", noaux_tc_topk);
  m.def("mm_w8a16_dq_forward(Tensor input, Tensor weight, Tensor scale, Tensor(a!) output, int blocksize) -> Tensor(a!)");
  m.def("mlp_w8a16_dq_forward(Tensor input, Tensor gate_weight, Tensor up_weight, Tensor down_weight, Tensor gate_scale, "
        "Tensor up_scale, Tensor down_scale, Tensor(a!) output, int blocksize) -> Tensor(a!)");
  m.def("enable_profile", enable_profile);
  m.def("disable_profile", disable_profile);
  m.def("_profile_report", _profile_report);
  m.def("_set_expert_numerics", _set_expert_numerics);
  m.def("_invalidate_weight_cache", _invalidate_weight_cache);
  m.def("_mm_weights(Tensor weight, Tensor scale) -> Tensor[]");
  m.def("_mlp_weights(Tensor gate_weight, Tensor up_weight, Tensor down_weight, Tensor gate_scale, Tensor up_scale, "
        "Tensor down_scale) -> Tensor[]");
  m.def("_layer_fp8(Tensor x, Tensor router_weight, Tensor w13, Tensor w13_scale, Tensor w2, Tensor w2_scale, int top_k, int mode, "
        "Tensor? bias, int n_groups, int topk_groups, bool renorm, float scale, Tensor? shared_w13, Tensor? shared_w13_scale, "
        "Tensor? shared_w2, Tensor? shared_w2_scale, Tensor(a!) out, Tensor(b!) workspace) -> int", _layer_fp8);
  m.def("_packed_weight_sets", _packed_weight_sets);
  m.def("_packed_weight_bytes", _packed_weight_bytes);
}

TORCH_LIBRARY_IMPL(my_ops, CompositeExplicitAutograd, m) {
  m.impl("mm_w8a16_dq_forward", mm_w8a16_dq_forward);
  m.impl("mlp_w8a16_dq_forward", mlp_w8a16_dq_forward);
  m.impl("_mm_weights", _mm_weights);
  m.impl("_mlp_weights", _mlp_weights);
}

}  // namespace at

// The eager read's autograd nodes, in C++ over the C ABI (attnres_hip.h).
//
// `attnres(values, query)` in eager mode (no dynamo tracing, plain tensors)
// calls `packed_read` / `sources_read` below instead of the torch.library
// ops, which remain the path under torch.compile.  Both launch the same
// kernels on the same saved state, so out, dv and dq are bit-identical
// between them.  What this file saves is host time: the node's forward and
// backward run without Python, and the backward -- which autograd runs on its
// device thread -- takes no Python lock.  On an MI355X box a small read
// (S = 8, N = 1024, D = 1024) costs 80 us of host time for forward plus
// torch.autograd.grad through these nodes, against 139 us through a Python
// autograd.Function, with torch's own floor for a trivial graph at 62 us.
// The packed node also flattens the batch axes itself (two view nodes less
// in the graph): c1's [8, 2, 512, 1024] read 37 us on a box whose floor is
// 29.5 us.  A read that needs no gradient skips the nodes (below).
//
// Saved state: the refinement bytes (when the read saves them) and the FP32
// statistics live in one byte allocation whose addresses are passed to the
// library (layout below), plus the inputs and, for a read that saves its
// refinement, the output.  Reference: the op pair it stands for,
// `attnres::_fixed_tail_forward_with_aux` / `_fixed_tail_backward`
// (fixed_tail.py:904-1034) and the source-list pair (fixed_tail_sources.py:
// 78-183); their autograd registration (fixed_tail.py:1041-1057): the aux
// outputs carry no gradient and a None upstream gradient gives None.

#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPStream.h>

#include <torch/csrc/autograd/graph_task.h>

#include <algorithm>
#include <memory>
#include <mutex>
#include <optional>
#include <vector>

#include "attnres_hip.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// A failing status raises as the Python binding does: ValueError for argument
// errors, RuntimeError otherwise, with the library's own message.
void check(int status, const char* what) {
  if (status == ATTNRES_OK) return;
  const char* message = attnres_hip_last_error();
  if (status == ATTNRES_ERR_SHAPE || status == ATTNRES_ERR_STRIDE || status == ATTNRES_ERR_SCALAR ||
      status == ATTNRES_ERR_WORKSPACE) {
    TORCH_CHECK_VALUE(false, what, ": ", message);
  }
  TORCH_CHECK(false, what, ": ", message, " (status ", status, ")");
}

// Pooled saved state: out_refine [N, D] int8 at byte 0 (when saved), then
// from the 16-byte aligned offset `head` logit [N, S], 1/rms [N, S] (`block`
// floats each) and stats [2, N], FP32; `size` bytes in all.  The Python
// `_pool_layout` states the same layout for the ops' pooled views.
struct PoolLayout {
  int64_t head, block, size;
};

PoolLayout pool_layout(int64_t tokens, int64_t sources, int64_t width, bool save) {
  const int64_t head = ((save ? tokens * width : 0) + 15) / 16 * 16;
  const int64_t block = tokens * sources;
  return {head, block, head + 4 * (2 * block + 2 * tokens)};
}

struct StatePointers {
  int8_t* refine;  // nullptr when the read saves no refinement
  float* logit;
  float* inv_rms;
  float* stats;
};

StatePointers pool_pointers(const Tensor& pool, const PoolLayout& layout, bool save) {
  char* base = static_cast<char*>(pool.data_ptr());
  float* logit = reinterpret_cast<float*>(base + layout.head);
  return {save ? reinterpret_cast<int8_t*>(base) : nullptr, logit, logit + layout.block, logit + 2 * layout.block};
}

hipStream_t current_stream(const Tensor& tensor) {
  return c10::hip::getCurrentHIPStream(tensor.device().index()).stream();
}

Tensor bf16_empty(at::IntArrayRef shape, const Tensor& like) {
  return torch::empty(shape, like.options().dtype(torch::kBFloat16));
}

Tensor dq_workspace(int64_t tokens, int64_t width, int64_t rank, const Tensor& like) {
  const int64_t elems = attnres_hip_dq_workspace_elems(tokens, width, rank);
  TORCH_CHECK_VALUE(elems >= 0, "attnres backward: shape outside the supported envelope");
  return torch::empty({elems}, like.options().dtype(torch::kFloat32));
}

// Element stride between consecutive rows of tensor[..., D] flattened to
// [rows, D], or nothing when the rows are not evenly spaced or a row is not
// unit-stride (the Python `row_stride`, after fla_full_sources.py:164-178).
std::optional<int64_t> row_stride(const Tensor& tensor) {
  const int64_t last = tensor.dim() - 1;
  if (tensor.size(last) > 1 && tensor.stride(last) != 1) return std::nullopt;
  std::optional<int64_t> stride;
  int64_t rows = 1;
  for (int64_t d = last - 1; d >= 0; --d) {
    if (tensor.size(d) == 1) continue;
    if (!stride) {
      stride = tensor.stride(d);
    } else if (tensor.stride(d) != rows * *stride) {
      return std::nullopt;
    }
    rows *= tensor.size(d);
  }
  return stride.value_or(0);
}

// Row pointers and strides of a source list; sources whose rows are not
// addressable are copied (the copies live until the launch is enqueued).
struct SourceTable {
  std::vector<Tensor> keep;
  std::vector<const void*> rows;
  std::vector<int64_t> strides;
};

SourceTable source_table(at::TensorList sources) {
  SourceTable table;
  table.keep.reserve(sources.size());
  for (const Tensor& source : sources) {
    Tensor rows = source;
    std::optional<int64_t> stride = row_stride(rows);
    if (!stride) {
      rows = rows.contiguous();
      stride = row_stride(rows);
    }
    table.keep.push_back(rows);
    table.rows.push_back(rows.data_ptr());
    table.strides.push_back(*stride);
  }
  return table;
}

int64_t rows_of(const Tensor& tensor) { return tensor.dim() > 1 ? tensor.numel() / tensor.size(-1) : 1; }

// Packed values [S, ..., D] as rows [S, N, D]: a view where the batch axes
// collapse to one row stride (as torch's reshape does), a copy otherwise, and
// a copy too when a row is not unit-stride.  Called inside a node's forward
// (or with no node at all), so autograd records no view nodes for it.
Tensor flat_rows(const Tensor& values) {
  const int64_t S = values.size(0), D = values.size(-1);
  Tensor rows = values.dim() == 3 ? values : values.reshape({S, -1, D});
  if (D > 1 && rows.stride(2) != 1) rows = rows.contiguous();
  return rows;
}

// ------------------------------------------------------------------ packed

struct PackedRead : public torch::autograd::Function<PackedRead> {
  // values [S, ..., D] (checked by the Python caller), query [R] contiguous.
  // The batch axes flatten to N rows here (flat_rows), so autograd records no
  // view nodes around the read: the output has the batch shape [..., D] and
  // the value gradient the shape of values.
  static Tensor forward(AutogradContext* ctx, const Tensor& values, const Tensor& query, double eps, double scale) {
    const int64_t S = values.size(0), D = values.size(-1), R = query.numel();
    const Tensor rows = flat_rows(values);
    const int64_t N = rows.size(1);
    const bool save = attnres_hip_saves_refinement_for(S, D, R) != 0;
    const c10::DeviceGuard guard(values.device());
    Tensor out = bf16_empty(values.sizes().slice(1), values);  // N contiguous rows
    const PoolLayout layout = pool_layout(N, S, D, save);
    Tensor pool = torch::empty({layout.size}, values.options().dtype(torch::kUInt8));
    const StatePointers state = pool_pointers(pool, layout, save);
    check(attnres_hip_packed_forward(rows.data_ptr(), rows.stride(0), rows.stride(1), S, N, D, query.data_ptr(), R,
                                     static_cast<float>(eps), static_cast<float>(scale), out.data_ptr(), state.refine,
                                     state.logit, state.inv_rms, state.stats, current_stream(values)),
          "attnres packed forward");
    ctx->set_materialize_grads(false);
    if (save) {
      ctx->save_for_backward({rows, query, pool, out});
    } else {
      ctx->save_for_backward({rows, query, pool});
    }
    ctx->saved_data["save"] = save;
    ctx->saved_data["scale"] = scale;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    const variable_list saved = ctx->get_saved_variables();
    const Tensor& rows = saved[0];  // [S, N, D]
    const Tensor& query = saved[1];
    const bool save = ctx->saved_data["save"].toBool();
    const int64_t S = rows.size(0), N = rows.size(1), D = rows.size(2), R = query.numel();
    const c10::DeviceGuard guard(rows.device());
    const Tensor grad_out = grads[0].to(torch::kBFloat16).contiguous();  // the output's shape [..., D]: N rows
    const Tensor out = save ? saved[3].contiguous() : Tensor();
    const StatePointers state = pool_pointers(saved[2], pool_layout(N, S, D, save), save);
    std::vector<int64_t> shape{S};  // the shape of values: [S] + the output's
    shape.insert(shape.end(), grad_out.sizes().begin(), grad_out.sizes().end());
    Tensor grad_values = bf16_empty(shape, rows);
    Tensor grad_query = bf16_empty({R}, rows);
    Tensor workspace = dq_workspace(N, D, R, rows);
    check(attnres_hip_packed_backward(rows.data_ptr(), rows.stride(0), rows.stride(1), S, N, D, query.data_ptr(), R,
                                      static_cast<float>(ctx->saved_data["scale"].toDouble()),
                                      save ? out.data_ptr() : nullptr, state.refine, grad_out.data_ptr(), state.logit,
                                      state.inv_rms, state.stats, grad_values.data_ptr(), grad_query.data_ptr(),
                                      workspace.data_ptr<float>(), workspace.numel(), current_stream(rows)),
          "attnres packed backward");
    return {ctx->needs_input_grad(0) ? grad_values : Tensor(), ctx->needs_input_grad(1) ? grad_query : Tensor(),
            Tensor(), Tensor()};
  }
};

// -------------------------------------------------------------------- list

struct SourcesRead : public torch::autograd::Function<SourcesRead> {
  // sources: S tensors [..., D] of one shape (checked by the Python caller);
  // each list position gets its own gradient.
  static Tensor forward(AutogradContext* ctx, const Tensor& query, double eps, double scale, at::TensorList sources) {
    const Tensor& first = sources[0];
    const int64_t S = static_cast<int64_t>(sources.size()), N = rows_of(first), D = first.size(-1);
    const int64_t R = query.numel();
    const bool save = attnres_hip_saves_refinement_for(S, D, R) != 0;
    const c10::DeviceGuard guard(first.device());
    const SourceTable table = source_table(sources);
    Tensor out = bf16_empty(first.sizes(), first);
    const PoolLayout layout = pool_layout(N, S, D, save);
    Tensor pool = torch::empty({layout.size}, first.options().dtype(torch::kUInt8));
    const StatePointers state = pool_pointers(pool, layout, save);
    check(attnres_hip_sources_forward(table.rows.data(), table.strides.data(), S, N, D, query.data_ptr(), R,
                                      static_cast<float>(eps), static_cast<float>(scale), out.data_ptr(), state.refine,
                                      state.logit, state.inv_rms, state.stats, current_stream(first)),
          "attnres source-list forward");
    ctx->set_materialize_grads(false);
    variable_list keep(sources.begin(), sources.end());
    keep.push_back(query);
    keep.push_back(pool);
    if (save) keep.push_back(out);
    ctx->save_for_backward(keep);
    ctx->saved_data["save"] = save;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["count"] = S;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const int64_t S = ctx->saved_data["count"].toInt();
    variable_list result(3 + S);  // query, eps, scale, then one per source
    if (!grads[0].defined()) return result;
    const variable_list saved = ctx->get_saved_variables();
    const std::vector<Tensor> sources(saved.begin(), saved.begin() + S);
    const Tensor& query = saved[S];
    const bool save = ctx->saved_data["save"].toBool();
    const Tensor& first = sources[0];
    const int64_t N = rows_of(first), D = first.size(-1), R = query.numel();
    const c10::DeviceGuard guard(first.device());
    const SourceTable table = source_table(sources);
    const Tensor grad_out = grads[0].to(torch::kBFloat16).contiguous();
    const Tensor out = save ? saved[S + 2].contiguous() : Tensor();
    const StatePointers state = pool_pointers(saved[S + 1], pool_layout(N, S, D, save), save);
    std::vector<Tensor> dv;
    std::vector<void*> dv_rows;
    dv.reserve(S);
    dv_rows.reserve(S);
    for (int64_t s = 0; s < S; ++s) {
      dv.push_back(bf16_empty(first.sizes(), first));
      dv_rows.push_back(dv.back().data_ptr());
    }
    Tensor grad_query = bf16_empty({R}, first);
    Tensor workspace = dq_workspace(N, D, R, first);
    check(attnres_hip_sources_backward(table.rows.data(), table.strides.data(), S, N, D, query.data_ptr(), R,
                                       static_cast<float>(ctx->saved_data["scale"].toDouble()),
                                       save ? out.data_ptr() : nullptr, state.refine, grad_out.data_ptr(), state.logit,
                                       state.inv_rms, state.stats, dv_rows.data(), grad_query.data_ptr(),
                                       workspace.data_ptr<float>(), workspace.numel(), current_stream(first)),
          "attnres source-list backward");
    if (ctx->needs_input_grad(0)) result[0] = grad_query;
    for (int64_t s = 0; s < S; ++s) {
      if (ctx->needs_input_grad(1 + s)) result[3 + s] = dv[s];
    }
    return result;
  }
};

// ------------------------------------------------------ no gradient needed

// Grad mode off (torch.no_grad, inference_mode) or no input requiring grad:
// no node, no saved state and no refinement bytes (the forward takes
// out_refine = NULL for any S); the statistics the kernels write go to a
// scratch allocation freed on return.  out is the same, bit for bit.
bool needs_grad(const Tensor& query, at::TensorList sources) {
  if (!at::GradMode::is_enabled()) return false;
  if (query.requires_grad()) return true;
  for (const Tensor& source : sources) {
    if (source.requires_grad()) return true;
  }
  return false;
}

Tensor statistics_scratch(int64_t tokens, int64_t sources, const Tensor& like, StatePointers* state) {
  const PoolLayout layout = pool_layout(tokens, sources, 0, false);
  Tensor pool = torch::empty({layout.size}, like.options().dtype(torch::kUInt8));
  *state = pool_pointers(pool, layout, false);
  return pool;
}

Tensor packed_forward_only(const Tensor& values, const Tensor& query, double eps, double scale) {
  const int64_t S = values.size(0), D = values.size(-1), R = query.numel();
  const Tensor rows = flat_rows(values);
  const int64_t N = rows.size(1);
  const c10::DeviceGuard guard(values.device());
  Tensor out = bf16_empty(values.sizes().slice(1), values);
  StatePointers state{};
  const Tensor scratch = statistics_scratch(N, S, values, &state);
  check(attnres_hip_packed_forward(rows.data_ptr(), rows.stride(0), rows.stride(1), S, N, D, query.data_ptr(), R,
                                   static_cast<float>(eps), static_cast<float>(scale), out.data_ptr(), nullptr,
                                   state.logit, state.inv_rms, state.stats, current_stream(values)),
        "attnres packed forward");
  return out;
}

Tensor sources_forward_only(const Tensor& query, double eps, double scale, at::TensorList sources) {
  const Tensor& first = sources[0];
  const int64_t S = static_cast<int64_t>(sources.size()), N = rows_of(first), D = first.size(-1);
  const c10::DeviceGuard guard(first.device());
  const SourceTable table = source_table(sources);
  Tensor out = bf16_empty(first.sizes(), first);
  StatePointers state{};
  const Tensor scratch = statistics_scratch(N, S, first, &state);
  check(attnres_hip_sources_forward(table.rows.data(), table.strides.data(), S, N, D, query.data_ptr(),
                                    query.numel(), static_cast<float>(eps), static_cast<float>(scale),
                                    out.data_ptr(), nullptr, state.logit, state.inv_rms, state.stats,
                                    current_stream(first)),
        "attnres source-list forward");
  return out;
}

Tensor packed_read(const Tensor& values, const Tensor& query, double eps, double scale) {
  if (!needs_grad(query, values)) return packed_forward_only(values, query, eps, scale);
  return PackedRead::apply(values, query, eps, scale);
}

Tensor sources_read(const Tensor& query, double eps, double scale, const std::vector<Tensor>& sources) {
  if (!needs_grad(query, sources)) return sources_forward_only(query, eps, scale, sources);
  return SourcesRead::apply(query, eps, scale, at::TensorList(sources));
}

// ------------------------------------------------------------- source bank

// The current stream of the tensor's device (as torch sees it: the stream an
// allocation made now belongs to).
c10::Stream stream_of(const Tensor& tensor) {
  return c10::impl::VirtualGuardImpl(tensor.device().type()).getStream(tensor.device());
}

// `tensor`, known to the allocator as used on stream `made`, is used by kernels
// of stream `now` (use_here: the current one): its memory is not handed out again before they end.
void use_on(const c10::Stream& now, const Tensor& tensor, const c10::Stream& made) {
  if (now != made) {
    c10::impl::VirtualGuardImpl(now.device_type()).recordDataPtrOnStream(tensor.storage().data_ptr(), now);
  }
}
void use_here(const Tensor& tensor, const c10::Stream& made) { use_on(stream_of(tensor), tensor, made); }

// The slots of a SourceBank and one backward pass's gradient bookkeeping,
// used by the nodes below (attnres/shared.py states the scheme).  The nodes
// hold it and it holds no token, so nothing closes a cycle.  Backward nodes
// run without Python's lock, possibly on several threads: `mutex` guards the
// pass's bookkeeping.  Pushes and reads may run on different streams: autograd
// orders their backward kernels (by the tokens), and what one node allocates and
// another uses is kept until that use ends (use_here).
struct BankState : public torch::CustomClassHolder {
  // One read's gathered terms: its dO, the query on row positions and the
  // coefficients [3, count, N]; kept until the gathers of its slots are enqueued.
  struct Record {
    Tensor grad_out, query_row, coef;
    int64_t count, rank;
    c10::Stream stream;  // of the read's backward
  };
  struct Pending {
    std::shared_ptr<Record> record;
    int64_t position;  // of the slot in the read's list
  };

  int64_t capacity;
  bool gather;       // gradients="gather", else accumulated FP32 sums
  bool bf16_gather;  // a BF16 source's gradient is stored as BF16 by its one gather launch
  Tensor values;     // [capacity, ..., D] BF16
  c10::Stream values_stream;
  int64_t tokens = 0, width = 0;

  std::mutex mutex;
  int64_t pass = -1;
  Tensor sums;  // [capacity, ..., D] FP32 (accumulate)
  std::optional<c10::Stream> sums_stream, sums_last;  // allocated on, last added to on
  std::vector<char> written;
  std::vector<std::vector<Pending>> pending;
  struct Partial {  // FP32 sums of a slot's earlier reads (gather_block)
    Tensor sum;
    std::optional<c10::Stream> stream;
  };
  std::vector<Partial> partial;

  // A slot's push node, whose first `inputs` edges lead to the slot's source (or
  // to the terms of its sum); empty when the push recorded none.  Weak: the node
  // holds this state.
  struct PushNode {
    std::weak_ptr<torch::autograd::Node> node;
    size_t inputs = 0;
  };
  std::vector<PushNode> push_nodes;

  BankState(int64_t capacity_, bool gather_, bool bf16_gather_, const Tensor& source)
      : capacity(capacity_), gather(gather_), bf16_gather(bf16_gather_), values_stream(stream_of(source)),
        written(capacity_, 0), pending(capacity_), partial(capacity_), push_nodes(capacity_) {
    std::vector<int64_t> shape{capacity};
    shape.insert(shape.end(), source.sizes().begin(), source.sizes().end());
    values = bf16_empty(shape, source);
    width = source.size(-1);
    tokens = source.numel() / width;
  }

  char* slot_rows(int64_t slot) const { return static_cast<char*>(values.data_ptr()) + slot * tokens * width * 2; }

  // The first read of a pass: nothing left from an earlier pass (one that
  // stopped short of the sources) is used, and sums handed out earlier stay
  // valid (fresh buffers).
  void begin_pass() {
    const int64_t current = torch::autograd::get_current_graph_task_id();
    if (pass == current) return;
    sums = Tensor();
    std::fill(written.begin(), written.end(), 0);
    for (auto& list : pending) list.clear();
    for (Partial& lower : partial) lower = Partial();
    pass = current;
  }

  // The current stream adds to the sums next, after what other streams added (no
  // autograd edge orders the backward kernels of two reads).
  void add_to_sums_here() {
    const c10::Stream now = stream_of(sums);
    if (now != *sums_last) {
      c10::Event added(now.device_type());
      added.record(*sums_last);
      added.block(now);
      sums_last = now;
    }
    use_on(now, sums, *sums_stream);
  }

  // Called by a Python thread, which lets go of its lock first: a backward call
  // may hold `mutex` and need that lock to free a tensor.
  void set_push_node(int64_t slot, const Tensor& token, size_t inputs) {
    const py::gil_scoped_release release;
    const std::lock_guard<std::mutex> lock(mutex);
    push_nodes[slot] = {token.grad_fn(), inputs};
  }

  // Whether the running backward pass computes a gradient for the slot's source.
  bool wanted(int64_t slot) const {
    const auto node = push_nodes[slot].node.lock();
    if (!node) return false;
    for (size_t i = 0; i < push_nodes[slot].inputs; ++i) {
      if (node->task_should_compute_output(i)) return true;
    }
    return false;
  }

  // A slot with many reads also forms the FP32 sums of the slots before it
  // over the same reads, whose dO rows are then read once for all of them; the
  // slots add what reads they get later to those sums.  Only where the reads
  // saw these slots one position apart (a Full schedule's prefixes) and the pass
  // computes their sources' gradients, so every sum is taken in this pass.  A block writes and reads 8 bytes of sums per
  // element and slot to save 2 per read, so it pays from about 9 reads on.
  bool gather_block(int64_t slot, const std::vector<Pending>& reads) const {
    if (reads.size() < kBlockReads || slot < ATTNRES_GATHER_SLOTS - 1) return false;
    for (int64_t k = 1; k < ATTNRES_GATHER_SLOTS; ++k) {
      const std::vector<Pending>& lower = pending[slot - k];
      if (!wanted(slot - k) || partial[slot - k].sum.defined() || lower.size() != reads.size()) return false;
      for (size_t i = 0; i < reads.size(); ++i) {
        if (lower[i].record != reads[i].record || lower[i].position != reads[i].position - k) return false;
      }
    }
    return true;
  }
  static constexpr size_t kBlockReads = 9;

  // Slot `slot`'s gradient for this pass, or an undefined tensor: gathered (in
  // BF16 when the source is BF16 and one launch covers the slot's reads, else
  // FP32), or a view of the FP32 accumulated sums.
  Tensor take(int64_t slot, at::ScalarType dtype) {
    const std::lock_guard<std::mutex> lock(mutex);
    if (pass != torch::autograd::get_current_graph_task_id()) return Tensor();
    if (!gather) {
      if (!written[slot]) return Tensor();
      written[slot] = 0;
      use_here(sums, *sums_stream);
      return sums.select(0, slot);
    }
    std::vector<Pending> reads;
    reads.swap(pending[slot]);
    Partial earlier;
    std::swap(earlier, partial[slot]);
    const Tensor base = earlier.sum;
    const c10::Stream now = stream_of(values);
    if (base.defined()) use_on(now, base, *earlier.stream);
    if (!wanted(slot)) return Tensor();
    // the sums of a block's slots lie in one allocation: an FP32 source receives a copy of its own
    const auto own = [&] { return base.defined() && dtype == torch::kFloat32 ? base.clone() : base; };
    if (reads.empty()) return own();
    use_on(now, values, values_stream);
    std::vector<attnres_gather_read> table;
    table.reserve(reads.size());
    bool one_launch = reads.size() <= ATTNRES_MAX_GATHER_READS;
    for (const Pending& p : reads) {
      const Record& r = *p.record;
      one_launch = one_launch && r.rank == reads[0].record->rank;
      for (const Tensor* term : {&r.grad_out, &r.query_row, &r.coef}) use_on(now, *term, r.stream);
      table.push_back({r.grad_out.data_ptr(), r.query_row.data_ptr(), r.coef.data_ptr<float>(), r.count, p.position,
                       r.rank});
    }
    const bool bf16 = one_launch && bf16_gather && dtype == torch::kBFloat16;
    const int grad_dtype = bf16 ? ATTNRES_DTYPE_BF16 : ATTNRES_DTYPE_F32;
    const auto count = static_cast<int64_t>(table.size());
    const c10::DeviceGuard guard(values.device());
    const auto fp32 = values.options().dtype(torch::kFloat32);
    if (!one_launch) {
      const bool add = base.defined();
      Tensor grad = add ? own() : torch::empty(values.sizes().slice(1), fp32);
      check(attnres_hip_bank_gather(slot_rows(slot), width, tokens, width, table.data(), count, grad.data_ptr(),
                                    grad_dtype, add ? 1 : 0, current_stream(values)),
            "attnres source-bank gather");
      return grad;
    }
    Tensor grad = torch::empty(values.sizes().slice(1), bf16 ? values.options() : fp32);
    const bool block = !base.defined() && gather_block(slot, reads);
    Tensor lower;  // [slots - 1, ..., D]
    if (block) {
      std::vector<int64_t> shape{ATTNRES_GATHER_SLOTS - 1};
      shape.insert(shape.end(), grad.sizes().begin(), grad.sizes().end());
      lower = torch::empty(shape, fp32);
    }
    check(attnres_hip_bank_gather_slots(slot_rows(slot), width, tokens * width, block ? ATTNRES_GATHER_SLOTS : 1,
                                        tokens, width, table.data(), count,
                                        base.defined() ? base.data_ptr<float>() : nullptr, grad.data_ptr(), grad_dtype,
                                        block ? lower.data_ptr<float>() : nullptr, current_stream(values)),
          "attnres source-bank gather");
    if (block) {
      for (int64_t k = 1; k < ATTNRES_GATHER_SLOTS; ++k) {
        partial[slot - k] = {lower.select(0, k - 1), now};
        pending[slot - k].clear();
      }
    }
    return grad;
  }
};

// Slots of a read: the leading `count`, then `tail` (-1: none).  Leading slots
// alone, or followed by the next one, are a prefix of the packed buffer.
struct Slots {
  int64_t count, tail;
  int64_t size() const { return count + (tail >= 0 ? 1 : 0); }
  int64_t at(int64_t i) const { return i < count ? i : tail; }
  bool prefix() const { return tail < 0 || tail == count; }
};

struct SlotTable {
  std::vector<const void*> rows;
  std::vector<int64_t> strides;
  SlotTable(const BankState& bank, const Slots& slots) : strides(slots.size(), bank.width) {
    for (int64_t i = 0; i < slots.size(); ++i) rows.push_back(bank.slot_rows(slots.at(i)));
  }
};

void bank_forward(const BankState& bank, const Slots& slots, const Tensor& query, double eps, double scale,
                  const Tensor& out, const StatePointers& state) {
  const int64_t S = slots.size(), N = bank.tokens, D = bank.width, R = query.numel();
  use_here(bank.values, bank.values_stream);
  if (slots.prefix()) {
    check(attnres_hip_packed_forward(bank.values.data_ptr(), N * D, D, S, N, D, query.data_ptr(), R,
                                     static_cast<float>(eps), static_cast<float>(scale), out.data_ptr(), state.refine,
                                     state.logit, state.inv_rms, state.stats, current_stream(bank.values)),
          "attnres packed forward");
  } else {
    const SlotTable table(bank, slots);
    check(attnres_hip_sources_forward(table.rows.data(), table.strides.data(), S, N, D, query.data_ptr(), R,
                                      static_cast<float>(eps), static_cast<float>(scale), out.data_ptr(), state.refine,
                                      state.logit, state.inv_rms, state.stats, current_stream(bank.values)),
          "attnres source-list forward");
  }
}

c10::intrusive_ptr<BankState> bank_of(AutogradContext* ctx) {
  return c10::static_intrusive_pointer_cast<BankState>(ctx->saved_data["bank"].toCapsule());
}

// The zero-size token that orders the nodes, and its zero-size gradient.
Tensor token_like(const Tensor& source) { return torch::empty({0}, source.options()); }

// Copy a source into its slot; the new token follows `previous` (the token of
// the push before; none for the first).
struct BankPush : public torch::autograd::Function<BankPush> {
  static Tensor forward(AutogradContext* ctx, const c10::intrusive_ptr<BankState>& bank, int64_t slot,
                        const Tensor& source, const std::optional<Tensor>& previous) {
    const c10::DeviceGuard guard(source.device());
    use_here(bank->values, bank->values_stream);
    bank->values.select(0, slot).copy_(source);
    ctx->set_materialize_grads(false);
    ctx->saved_data["bank"] = c10::IValue::make_capsule(bank);
    ctx->saved_data["slot"] = slot;
    ctx->saved_data["dtype"] = static_cast<int64_t>(source.scalar_type());
    ctx->saved_data["token"] = previous.has_value();
    return token_like(source);
  }

  static variable_list backward(AutogradContext* ctx, variable_list) {
    const auto bank = bank_of(ctx);
    const auto dtype = static_cast<at::ScalarType>(ctx->saved_data["dtype"].toInt());
    Tensor grad = bank->take(ctx->saved_data["slot"].toInt(), dtype);
    if (grad.defined()) grad = grad.to(dtype);
    const bool token = ctx->saved_data["token"].toBool();
    return {Tensor(), Tensor(), grad, token ? torch::empty({0}, bank->values.options().dtype(dtype)) : Tensor()};
  }
};

// partial = prev + emitted, with its BF16 copy written into the slot by the
// same kernel; the gradient of both inputs is that of the partial plus the
// slot's summed read gradient.
struct BankPushSum : public torch::autograd::Function<BankPushSum> {
  static variable_list forward(AutogradContext* ctx, const c10::intrusive_ptr<BankState>& bank, int64_t slot,
                               const Tensor& prev, const Tensor& emitted, const std::optional<Tensor>& previous) {
    const c10::DeviceGuard guard(emitted.device());
    const Tensor a = prev.contiguous(), b = emitted.contiguous();
    Tensor partial = torch::empty(b.sizes(), b.options());
    use_here(bank->values, bank->values_stream);
    check(attnres_hip_partial_sum(a.data_ptr(), b.data_ptr(),
                                  b.scalar_type() == torch::kFloat32 ? ATTNRES_DTYPE_F32 : ATTNRES_DTYPE_BF16,
                                  b.numel(), partial.data_ptr(), bank->slot_rows(slot), current_stream(b)),
          "attnres partial sum");
    ctx->set_materialize_grads(false);
    ctx->saved_data["bank"] = c10::IValue::make_capsule(bank);
    ctx->saved_data["slot"] = slot;
    ctx->saved_data["dtype"] = static_cast<int64_t>(emitted.scalar_type());
    ctx->saved_data["token"] = previous.has_value();
    return {partial, token_like(emitted)};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto bank = bank_of(ctx);
    const auto dtype = static_cast<at::ScalarType>(ctx->saved_data["dtype"].toInt());
    Tensor grad = bank->take(ctx->saved_data["slot"].toInt(), dtype);
    if (grad.defined()) grad = grad.to(dtype);
    if (grads[0].defined()) grad = grad.defined() ? grads[0] + grad : grads[0];
    // neither the partial nor the slot was used: a zero gradient, not an absent one
    if (!grad.defined() && (ctx->needs_input_grad(0) || ctx->needs_input_grad(1))) {
      grad = torch::zeros(bank->values.sizes().slice(1), bank->values.options().dtype(dtype));
    }
    const bool token = ctx->saved_data["token"].toBool();
    return {Tensor(), Tensor(), grad, grad, token ? torch::empty({0}, bank->values.options().dtype(dtype)) : Tensor()};
  }
};

// A read of the bank's slots.  Always saves the refinement (its backward
// kernels read it); the backward leaves dv to the slots' gathers, or adds it
// to their FP32 sums.  A read whose output received no gradient counts as one
// with a zero gradient: its query and sources get zeros, not nothing.
struct BankRead : public torch::autograd::Function<BankRead> {
  static Tensor forward(AutogradContext* ctx, const c10::intrusive_ptr<BankState>& bank, int64_t count, int64_t tail,
                        const Tensor& query, double eps, double scale, const Tensor& token) {
    const Slots slots{count, tail};
    const c10::DeviceGuard guard(bank->values.device());
    const Tensor q = query.contiguous();
    Tensor out = bf16_empty(bank->values.sizes().slice(1), bank->values);
    const PoolLayout layout = pool_layout(bank->tokens, slots.size(), bank->width, true);
    Tensor pool = torch::empty({layout.size}, bank->values.options().dtype(torch::kUInt8));
    bank_forward(*bank, slots, q, eps, scale, out, pool_pointers(pool, layout, true));
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, pool, out});
    ctx->saved_data["bank"] = c10::IValue::make_capsule(bank);
    ctx->saved_data["count"] = count;
    ctx->saved_data["tail"] = tail;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["dtype"] = static_cast<int64_t>(token.scalar_type());
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list result(7);  // bank, count, tail, query, eps, scale, token
    const auto bank = bank_of(ctx);
    const Slots slots{ctx->saved_data["count"].toInt(), ctx->saved_data["tail"].toInt()};
    const float scale = static_cast<float>(ctx->saved_data["scale"].toDouble());
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &query = saved[0], &pool = saved[1], out = saved[2].contiguous();
    const Tensor& like = bank->values;
    const int64_t S = slots.size(), N = bank->tokens, D = bank->width, R = query.numel();
    const c10::DeviceGuard guard(like.device());
    const Tensor grad_out = grads[0].defined() ? grads[0].to(torch::kBFloat16).contiguous()
                                               : torch::zeros(like.sizes().slice(1), like.options());
    const StatePointers state = pool_pointers(pool, pool_layout(N, S, D, true), true);
    Tensor grad_query = bf16_empty({R}, like);
    Tensor workspace = dq_workspace(N, D, R, like);
    const auto stream = current_stream(like);
    use_here(like, bank->values_stream);
    const std::lock_guard<std::mutex> lock(bank->mutex);
    bank->begin_pass();
    if (bank->gather) {
      Tensor coef = torch::empty({3, S, N}, like.options().dtype(torch::kFloat32));
      if (slots.prefix()) {
        check(attnres_hip_packed_backward_coef(like.data_ptr(), N * D, D, S, N, D, query.data_ptr(), R, scale,
                                               out.data_ptr(), state.refine, grad_out.data_ptr(), state.logit,
                                               state.inv_rms, state.stats, coef.data_ptr<float>(),
                                               grad_query.data_ptr(), workspace.data_ptr<float>(), workspace.numel(),
                                               stream),
              "attnres source-bank coefficient backward");
      } else {
        const SlotTable table(*bank, slots);
        check(attnres_hip_sources_backward_coef(table.rows.data(), table.strides.data(), S, N, D, query.data_ptr(), R,
                                                scale, out.data_ptr(), state.refine, grad_out.data_ptr(), state.logit,
                                                state.inv_rms, state.stats, coef.data_ptr<float>(),
                                                grad_query.data_ptr(), workspace.data_ptr<float>(),
                                                workspace.numel(), stream),
              "attnres source-bank coefficient backward");
      }
      Tensor query_row = query;
      if (R != D) {  // the query on the row's last R elements, zeros before
        query_row = torch::zeros({D}, query.options());
        query_row.narrow(0, D - R, R).copy_(query);
      }
      const auto record = std::make_shared<BankState::Record>(
          BankState::Record{grad_out, query_row, coef, S, R, stream_of(like)});
      for (int64_t i = 0; i < S; ++i) bank->pending[slots.at(i)].push_back({record, i});
    } else {
      if (!bank->sums.defined()) {
        bank->sums = torch::empty(like.sizes(), like.options().dtype(torch::kFloat32));
        bank->sums_stream = bank->sums_last = stream_of(like);
      }
      bank->add_to_sums_here();
      std::vector<uint8_t> flags;
      for (int64_t i = 0; i < S; ++i) flags.push_back(bank->written[slots.at(i)] ? 1 : 0);
      float* sums = bank->sums.data_ptr<float>();
      if (slots.prefix()) {
        check(attnres_hip_packed_backward_accumulate_f32(
                  like.data_ptr(), N * D, D, S, N, D, query.data_ptr(), R, scale, out.data_ptr(), state.refine,
                  grad_out.data_ptr(), state.logit, state.inv_rms, state.stats, sums, grad_query.data_ptr(),
                  workspace.data_ptr<float>(), workspace.numel(), flags.data(), stream),
              "attnres source-bank backward");
      } else {
        const SlotTable table(*bank, slots);
        std::vector<float*> rows;
        for (int64_t i = 0; i < S; ++i) rows.push_back(sums + slots.at(i) * N * D);
        check(attnres_hip_sources_backward_accumulate_f32(
                  table.rows.data(), table.strides.data(), S, N, D, query.data_ptr(), R, scale, out.data_ptr(),
                  state.refine, grad_out.data_ptr(), state.logit, state.inv_rms, state.stats, rows.data(),
                  grad_query.data_ptr(), workspace.data_ptr<float>(), workspace.numel(), flags.data(), stream),
              "attnres source-bank backward");
      }
      for (int64_t i = 0; i < S; ++i) bank->written[slots.at(i)] = 1;
    }
    if (ctx->needs_input_grad(0)) result[3] = grad_query;
    result[6] = torch::empty({0}, like.options().dtype(static_cast<at::ScalarType>(ctx->saved_data["dtype"].toInt())));
    return result;
  }
};

// The token after a push: with grad mode off it is the one before, so that later
// reads still order themselves after (and reach) the pushes that want gradients.
Tensor next_token(const Tensor& token, const std::optional<Tensor>& previous) {
  return !token.requires_grad() && previous && previous->requires_grad() ? *previous : token;
}

Tensor bank_push(const c10::intrusive_ptr<BankState>& bank, int64_t slot, const Tensor& source,
                 const std::optional<Tensor>& previous) {
  Tensor token = BankPush::apply(bank, slot, source, previous);
  bank->set_push_node(slot, token, 1);
  return next_token(token, previous);
}

std::tuple<Tensor, Tensor> bank_push_sum(const c10::intrusive_ptr<BankState>& bank, int64_t slot, const Tensor& prev,
                                         const Tensor& emitted, const std::optional<Tensor>& previous) {
  const variable_list results = BankPushSum::apply(bank, slot, prev, emitted, previous);
  bank->set_push_node(slot, results[1], 2);
  return {results[0], next_token(results[1], previous)};
}

// No gradient wanted (grad mode off, or neither the query nor the sources --
// through the token -- require one): the forward alone, nothing saved.
Tensor bank_read(const c10::intrusive_ptr<BankState>& bank, int64_t count, int64_t tail, const Tensor& query,
                 double eps, double scale, const Tensor& token) {
  if (at::GradMode::is_enabled() && (query.requires_grad() || token.requires_grad())) {
    return BankRead::apply(bank, count, tail, query, eps, scale, token);
  }
  const Slots slots{count, tail};
  const c10::DeviceGuard guard(bank->values.device());
  Tensor out = bf16_empty(bank->values.sizes().slice(1), bank->values);
  StatePointers state{};
  const Tensor scratch = statistics_scratch(bank->tokens, slots.size(), bank->values, &state);
  bank_forward(*bank, slots, query.contiguous(), eps, scale, out, state);
  return out;
}

std::tuple<int64_t, int64_t, int64_t> layout_of(int64_t tokens, int64_t sources, int64_t width, bool save) {
  const PoolLayout layout = pool_layout(tokens, sources, width, save);
  return {layout.head, layout.block, layout.size};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "Eager autograd nodes of the attnres read over the attnres_hip C ABI";
  m.def("packed_read", &packed_read, "packed read [S, ..., D] (eager autograd node)");
  m.def("sources_read", &sources_read, "source-list read (eager autograd node)");
  py::class_<BankState, c10::intrusive_ptr<BankState>>(m, "BankState", "the slots of a SourceBank")
      .def(py::init<int64_t, bool, bool, const Tensor&>())
      .def_readonly("_values", &BankState::values);
  m.def("bank_push", &bank_push, "copy a source into its slot; returns the new token");
  m.def("bank_push_sum", &bank_push_sum, "partial sum of a block, stored in a slot; returns it and the new token");
  m.def("bank_read", &bank_read, "read of leading slots and a tail slot (-1: none)");
  m.def("pool_layout", &layout_of, "(head, block, size) of the pooled saved state");
}

// The autograd functions behind kraken_amd/torch_embedding.py, over the C ABI.
//
// A step of an embedding layer is two or three kernel launches of a few microseconds each, so what
// the host does around them is what a small or ordinary batch waits for. As
// torch.autograd.Function classes in Python (pytorch/embedding.py:9-23,
// pytorch/combine_embedding.py:10-31 in the reference) a forward and a backward of one layer cost
// 60 to 120 us, most of it interpreter work and the hand-over of the interpreter lock to the
// engine's thread and back; 26 tables cost 400 us. Here a forward is one call that builds the
// request from the tensors' addresses, and the backward node runs in the engine's thread without
// taking the lock.
//
// Tensors are used where they lie: the ids of a combined request are not concatenated, and a
// gradient that is a block of columns of a wider matrix (what torch.cat along the feature dimension
// hands back) is read in place.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <memory>
#include <mutex>
#include <vector>

#include "kraken_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::edge_list;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

constexpr uint32_t kFlags = KRK_DEVICE_PTRS | KRK_ASYNC;

// api.KrakenHipError, as the ctypes calls raise it; usable with and without the interpreter lock.
[[noreturn]] void fail(int32_t rc, const char* what) {
  py::gil_scoped_acquire gil;
  py::object type = py::module_::import("kraken_amd.api").attr("KrakenHipError");
  py::object err = type(rc, what);
  PyErr_SetObject(type.ptr(), err.ptr());
  python_error e;
  e.persist();
  throw e;
}
#define KRK_CALL(fn, ...)                       \
  do {                                          \
    const int32_t rc_ = fn(__VA_ARGS__);        \
    if (rc_ != KRK_SUCCESS) fail(rc_, #fn);     \
  } while (0)

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// int64 ids are the uint64 ids bit for bit (worker/emitter.cc:126 casts the same way)
Tensor ids_of(const Tensor& t, const char* name = "indices") {
  if (t.scalar_type() != at::kLong || !t.is_cuda()) {
    throw py::type_error(std::string(name) + " must be an int64 CUDA tensor");
  }
  return t.contiguous();
}
const uint64_t* id_ptr(const Tensor& t) { return reinterpret_cast<const uint64_t*>(t.const_data_ptr<int64_t>()); }
const int64_t* off_ptr(const Tensor& t) { return t.const_data_ptr<int64_t>(); }
const float* float_ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr<float>() : nullptr; }

Tensor weights_of(const c10::optional<Tensor>& w) {
  return w.has_value() && w->defined() ? w->detach().contiguous().to(at::kFloat) : Tensor();
}

Tensor new_rows(at::IntArrayRef sizes, const Tensor& like) {
  return at::empty(sizes, at::TensorOptions().dtype(at::kFloat).device(like.device()));
}

Tensor new_zeros(at::IntArrayRef sizes, const Tensor& like) {
  return at::zeros(sizes, at::TensorOptions().dtype(at::kFloat).device(like.device()));
}

// `g` as `n` whole rows of `dim` floats one after the other, where the kernels' 16-byte loads may take
// them; zeros where a function behind the output had no gradient to hand on. A contiguous tensor need not start on 16 bytes: a row that torch.cat hands back behind 13
// dense features lies 52 bytes into theirs, and contiguous() returns it as it is.
Tensor dense_rows(const Tensor& g, int64_t n, int64_t dim, const Tensor& like) {
  if (!g.defined()) return new_zeros({n, dim}, like);
  Tensor rows = g.contiguous().to(at::kFloat);
  const bool vec = dim % 4 == 0;
  if (vec && (reinterpret_cast<uintptr_t>(rows.const_data_ptr<float>()) & 15) != 0) rows = rows.clone();
  return rows;
}

// The gradient rows of `g` where they lie, `stride` floats apart, if the kernels can read them there;
// otherwise of a dense float copy. `keep` holds whichever it is.
struct Rows {
  Tensor keep;
  int64_t stride = 0;
  float* ptr() const { return const_cast<float*>(keep.const_data_ptr<float>()); }
};
Rows rows_of(const Tensor& g, int64_t dim) {
  Rows r;
  r.stride = dim;
  if (g.scalar_type() == at::kFloat && g.dim() >= 1 && g.size(-1) == dim && (dim == 1 || g.stride(-1) == 1)) {
    int64_t stride = -1, span = 0;
    bool ok = true;
    for (int64_t i = g.dim() - 2; i >= 0 && ok; --i) {
      if (g.size(i) == 1) continue;
      if (stride < 0) {
        stride = g.stride(i);
        span = stride * g.size(i);
      } else {
        ok = g.stride(i) == span;
        span *= g.size(i);
      }
    }
    if (stride < 0) stride = dim;
    const bool vec = dim % 4 == 0;
    ok = ok && stride < ((int64_t)1 << 30) &&
         (!vec || (stride % 4 == 0 && (reinterpret_cast<uintptr_t>(g.const_data_ptr<float>()) & 15) == 0));
    if (ok) {
      r.keep = g;
      r.stride = stride;
      return r;
    }
  }
  r.keep = dense_rows(g, g.numel() / dim, dim, g);
  return r;
}

// The gradient rows of an output the loss never used: one row of zeros that every position reads. The
// rows still take their step with it (moments decay, counters advance, weights decay).
Rows zero_rows(const Tensor& like, int64_t dim) {
  Rows r;
  r.keep = new_zeros({dim}, like);
  return r;
}

// Whether a backward may use the rows that its forward's pull noted: it pushes for the very buffer that
// was pulled from. Saved-tensor hooks hand back a tensor of their own, and one that offloads may bring
// the ids of one pass to where the ids of a later pass were noted.
uint32_t as_pulled(const SavedVariable& ids) { return ids.has_hooks() ? 0u : KRK_IDS_AS_PULLED; }
uint32_t as_pulled(const std::vector<SavedVariable>& ids) {
  for (const SavedVariable& v : ids)
    if (v.has_hooks()) return 0u;
  return KRK_IDS_AS_PULLED;
}

bool recording(const Tensor& param) { return at::GradMode::is_enabled() && param.requires_grad(); }

// The node of a pass over `param` (the empty Parameter that stands for the tables, whose edge is
// what makes the engine run the node).
template <typename N>
std::shared_ptr<N> new_node(const Tensor& param) {
  auto node = std::shared_ptr<N>(new N(), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(param));
  return node;
}

// ---- what the Python side owns ------------------------------------------------------------------
// A value inside a ctypes object (a handle's c_void_p, an optimizer's struct). The object is kept as
// long as it is bound, so the address stays good whatever becomes of the Python objects around it;
// its owner may change the value, or bind another object, at any time (api.SparseTable.close() stores
// a null handle, which the C ABI answers with an error). Reading takes no interpreter lock: the
// value is copied under a lock of its own.
template <typename T>
class Bound {
 public:
  explicit Bound(const py::object& o) : object_(o), value_(address(o)) {}
  ~Bound() {
    if (!Py_IsInitialized()) {
      (void)object_.release();
      return;
    }
    py::gil_scoped_acquire gil;      // the last node of a graph dies in the engine's thread
    object_ = py::object();
  }
  Bound(const Bound&) = delete;
  Bound& operator=(const Bound&) = delete;
  T get() const {
    std::lock_guard<std::mutex> lk(mu_);
    return *value_;
  }
  void bind(py::object o) {          // the caller holds the interpreter lock; `o` leaves with the old object
    T* value = address(o);
    std::lock_guard<std::mutex> lk(mu_);
    std::swap(object_, o);
    value_ = value;
  }

 private:
  static T* address(const py::object& o) {
    return reinterpret_cast<T*>(py::module_::import("ctypes").attr("addressof")(o).cast<uintptr_t>());
  }
  mutable std::mutex mu_;
  py::object object_;
  T* value_;
};

// ---- one table --------------------------------------------------------------------------------
struct Table {
  Bound<krk_sparse*> h;
  Bound<krk_optim> optim;
  int64_t dim;
  double lr;
};
using TablePtr = std::shared_ptr<Table>;

struct EmbeddingBackward : Node {
  TablePtr table;
  SavedVariable ids;
  variable_list apply(variable_list&& grads) override {
    const Tensor saved = ids.unpack();
    const Tensor g = dense_rows(grads[0], saved.numel(), table->dim, saved);
    krk_sparse* h = table->h.get();
    const krk_optim optim = table->optim.get();
    KRK_CALL(krk_sparse_set_stream, h, current_stream());
    KRK_CALL(krk_sparse_push_raw, h, &optim, id_ptr(saved), saved.numel(), float_ptr(g), table->dim,
             (float)table->lr, kFlags | as_pulled(ids));
    return variable_list(1);
  }
  void release_variables() override { ids.reset_data(); }
  std::string name() const override { return "EmbeddingFunctionBackward"; }
};

Tensor embedding(const TablePtr& table, const Tensor& param, const Tensor& indices) {
  const Tensor ids = ids_of(indices);
  std::vector<int64_t> sizes = indices.sizes().vec();
  sizes.push_back(table->dim);
  Tensor out = new_rows(sizes, ids);
  const bool record = recording(param);
  krk_sparse* h = table->h.get();
  KRK_CALL(krk_sparse_set_stream, h, current_stream());
  // the table notes where it found every id: backward pushes gradients for this very tensor
  // (autograd keeps it alive and unchanged), so its look-up need not be repeated
  KRK_CALL(krk_sparse_pull, h, id_ptr(ids), ids.numel(), out.mutable_data_ptr<float>(),
           kFlags | (record ? KRK_NOTE_ROWS : 0u));
  if (record) {
    auto node = new_node<EmbeddingBackward>(param);
    node->table = table;
    node->ids = SavedVariable(ids, false);
    torch::autograd::set_history(out, node);
  }
  return out;
}

struct JaggedBackward : Node {
  TablePtr table;
  int mode = 0;
  SavedVariable ids, offsets;
  Tensor weights;
  variable_list apply(variable_list&& grads) override {
    const Tensor saved = ids.unpack(), off = offsets.unpack();
    const Tensor g = dense_rows(grads[0], off.numel() - 1, table->dim, saved);
    krk_sparse* h = table->h.get();
    const krk_optim optim = table->optim.get();
    KRK_CALL(krk_sparse_set_stream, h, current_stream());
    KRK_CALL(krk_sparse_push_pooled, h, &optim, id_ptr(saved), saved.numel(), off_ptr(off),
             off.numel() - 1, float_ptr(weights), mode, float_ptr(g), table->dim, (float)table->lr,
             kFlags | as_pulled(ids));
    return variable_list(1);
  }
  void release_variables() override {
    ids.reset_data();
    offsets.reset_data();
    weights.reset();
  }
  std::string name() const override { return "JaggedEmbeddingFunctionBackward"; }
};

Tensor jagged(const TablePtr& table, const Tensor& param, const Tensor& indices, const Tensor& offsets_in,
              const c10::optional<Tensor>& weights_in, int mode, double patch) {
  const Tensor ids = ids_of(indices);
  const Tensor off = ids_of(offsets_in, "offsets");
  const Tensor w = weights_of(weights_in);
  const int64_t bags = off.numel() - 1;
  Tensor out = new_rows({bags, table->dim}, ids);
  const bool record = recording(param);
  krk_sparse* h = table->h.get();
  KRK_CALL(krk_sparse_set_stream, h, current_stream());
  KRK_CALL(krk_sparse_pull_pooled, h, id_ptr(ids), ids.numel(), off_ptr(off), bags, float_ptr(w), mode,
           (float)patch, out.mutable_data_ptr<float>(), kFlags | (record ? KRK_NOTE_ROWS : 0u));
  if (record) {
    auto node = new_node<JaggedBackward>(param);
    node->table = table;
    node->mode = mode;
    node->ids = SavedVariable(ids, false);
    node->offsets = SavedVariable(off, false);
    node->weights = w;
    torch::autograd::set_history(out, node);
  }
  return out;
}

// ---- the tables of a combined request -----------------------------------------------------------
// Tables of equal dimension form one group of the engine; mixed dimensions give several groups.
struct Combine {
  struct Group {
    std::unique_ptr<Bound<krk_group*>> h;
    int64_t dim;
    std::vector<int> members;      // positions of its tables in the request
  };
  std::vector<Group> groups;
  std::vector<std::unique_ptr<Bound<krk_sparse*>>> tables;
  std::vector<int64_t> dims;
  Bound<krk_optim> optim;
  double lr;
  int64_t combined_max = (int64_t)1 << 28;   // groups whose pooled request is larger are served a table at a time
};
using CombinePtr = std::shared_ptr<Combine>;

// Piece `sizes` of a storage that several outputs share, `at` floats from its start: a tensor of its
// own (the pieces do not overlap, so none is a view of another).
Tensor piece_of(const Tensor& whole, int64_t at, at::IntArrayRef sizes) {
  Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(whole.storage()), whole.key_set(), whole.dtype());
  t.unsafeGetTensorImpl()->set_storage_offset(at);
  t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
  return t;
}

struct CombineBackward : Node {
  CombinePtr c;
  std::vector<SavedVariable> ids;
  variable_list apply(variable_list&& grads) override {
    void* stream = current_stream();
    const krk_optim optim = c->optim.get();
    const uint32_t noted = as_pulled(ids);
    for (const Combine::Group& g : c->groups) {
      krk_group* h = g.h->get();
      std::vector<krk_part> parts(g.members.size());
      std::vector<Tensor> keep;
      keep.reserve(2 * g.members.size());
      Rows zeros;
      for (size_t m = 0; m < g.members.size(); ++m) {
        const int i = g.members[m];
        Tensor saved = ids[i].unpack();
        krk_part& p = parts[m];
        p.ids = id_ptr(saved);
        p.n = saved.numel();
        if (grads[i].defined()) {
          Rows r = rows_of(grads[i], g.dim);
          p.rows = r.ptr();
          p.stride = r.stride;
          keep.push_back(std::move(r.keep));
        } else {
          if (!zeros.keep.defined()) zeros = zero_rows(saved, g.dim);
          p.rows = zeros.ptr();
          p.stride = zeros.stride;
        }
        keep.push_back(std::move(saved));
      }
      KRK_CALL(krk_group_set_stream, h, stream);
      KRK_CALL(krk_group_push_raw_parts, h, &optim, parts.data(), g.dim, (float)c->lr, kFlags | noted);
    }
    return variable_list(1);
  }
  void release_variables() override {
    for (auto& v : ids) v.reset_data();
  }
  std::string name() const override { return "CombineEmbeddingFunctionBackward"; }
};

std::vector<Tensor> combine(const CombinePtr& c, const Tensor& param, const std::vector<Tensor>& indices) {
  if (indices.size() != c->dims.size()) throw py::value_error("one index tensor per table");
  const bool record = recording(param);
  void* stream = current_stream();
  std::vector<Tensor> outs(indices.size()), ids(indices.size());
  std::vector<int64_t> sizes;
  for (const Combine::Group& g : c->groups) {
    std::vector<krk_part> parts(g.members.size());
    int64_t total = 0;
    for (int i : g.members) {
      ids[i] = ids_of(indices[i]);
      total += ids[i].numel();
    }
    const Tensor whole = new_rows({total, g.dim}, ids[g.members[0]]);
    float* base = whole.mutable_data_ptr<float>();
    int64_t at = 0;
    for (size_t m = 0; m < g.members.size(); ++m) {
      const int i = g.members[m];
      sizes.assign(indices[i].sizes().begin(), indices[i].sizes().end());
      sizes.push_back(g.dim);
      outs[i] = piece_of(whole, at, sizes);
      parts[m] = krk_part{id_ptr(ids[i]), ids[i].numel(), base + at, g.dim};
      at += ids[i].numel() * g.dim;
    }
    krk_group* h = g.h->get();
    KRK_CALL(krk_group_set_stream, h, stream);
    KRK_CALL(krk_group_pull_parts, h, parts.data(), kFlags | (record ? KRK_NOTE_ROWS : 0u));
  }
  if (record) {
    auto node = new_node<CombineBackward>(param);
    node->c = c;
    node->ids.reserve(ids.size());
    for (const Tensor& t : ids) node->ids.emplace_back(t, false);
    for (Tensor& o : outs) torch::autograd::set_history(o, node);
  }
  return outs;
}

// A pooled request is made of the tables' own calls: one whose table was closed is refused, also where
// the group still holds the table.
void check_open(const Combine& c) {
  for (const auto& t : c.tables)
    if (!t->get()) KRK_CALL(krk_sparse_sync, nullptr);
}

struct CombineJaggedBackward : Node {
  CombinePtr c;
  bool combined = true;            // every group's pull was one request, which noted its rows
  std::vector<int> modes;
  std::vector<SavedVariable> ids, offsets;
  std::vector<Tensor> weights;
  variable_list apply(variable_list&& grads) override {
    void* stream = current_stream();
    const krk_optim optim = c->optim.get();
    const uint32_t noted = combined ? as_pulled(ids) : 0u;
    check_open(*c);
    for (const Combine::Group& g : c->groups) {
      krk_group* h = g.h->get();
      std::vector<krk_pooled_part> parts(g.members.size());
      std::vector<Tensor> keep;
      keep.reserve(3 * g.members.size());
      Rows zeros;
      int64_t total = 0;
      for (size_t m = 0; m < g.members.size(); ++m) {
        const int i = g.members[m];
        krk_pooled_part& p = parts[m];
        p = krk_pooled_part{};
        Tensor saved = ids[i].unpack(), off = offsets[i].unpack();
        p.ids = id_ptr(saved);
        p.n = saved.numel();
        p.offsets = off_ptr(off);
        p.bags = off.numel() - 1;
        p.weights = float_ptr(weights[i]);
        p.mode = modes[i];
        if (grads[i].defined()) {
          Rows r = rows_of(grads[i], g.dim);
          p.rows = r.ptr();
          p.stride = r.stride;
          keep.push_back(std::move(r.keep));
        } else {
          if (!zeros.keep.defined()) zeros = zero_rows(saved, g.dim);
          p.rows = zeros.ptr();
          p.stride = zeros.stride;
        }
        total += std::max(p.n, p.bags);
        keep.push_back(std::move(saved));
        keep.push_back(std::move(off));
      }
      KRK_CALL(krk_group_set_stream, h, stream);
      const int32_t rc = total > c->combined_max
                             ? KRK_E_CAPACITY
                             : krk_group_push_pooled_parts(h, &optim, parts.data(), g.dim, (float)c->lr,
                                                           kFlags | noted);
      if (rc == KRK_SUCCESS) continue;
      if (rc != KRK_E_CAPACITY) fail(rc, "krk_group_push_pooled_parts");
      // more than one launch can name: a table at a time
      for (size_t m = 0; m < g.members.size(); ++m) {
        const krk_pooled_part& p = parts[m];
        if (p.n == 0 || p.bags == 0) continue;
        const int i = g.members[m];
        // a call of its own takes a row a bag
        const Tensor rows = dense_rows(grads[i], p.bags, g.dim, keep[0]);
        KRK_CALL(krk_sparse_push_pooled, c->tables[i]->get(), &optim, p.ids, p.n, p.offsets, p.bags, p.weights,
                 p.mode, float_ptr(rows), g.dim, (float)c->lr, kFlags);
      }
    }
    return variable_list(1);
  }
  void release_variables() override {
    for (auto& v : ids) v.reset_data();
    for (auto& v : offsets) v.reset_data();
    weights.clear();
  }
  std::string name() const override { return "CombineJaggedEmbeddingFunctionBackward"; }
};

std::vector<Tensor> combine_jagged(const CombinePtr& c, const Tensor& param, const std::vector<int>& modes,
                                   const std::vector<double>& patches, const std::vector<Tensor>& values,
                                   const std::vector<Tensor>& offsets_in,
                                   const std::vector<c10::optional<Tensor>>& weights_in) {
  const size_t n = c->tables.size();
  if (values.size() != n || offsets_in.size() != n || weights_in.size() != n || modes.size() != n ||
      patches.size() != n)
    throw py::value_error("one jagged batch per table");
  const bool record = recording(param);
  void* stream = current_stream();
  check_open(*c);
  bool combined = true;
  std::vector<Tensor> outs(n), ids(n), offsets(n), weights(n);
  for (const Combine::Group& g : c->groups) {
    std::vector<krk_pooled_part> parts(g.members.size());
    int64_t total = 0, bags = 0;
    for (int i : g.members) {
      ids[i] = ids_of(values[i]);
      offsets[i] = ids_of(offsets_in[i], "offsets");
      weights[i] = weights_of(weights_in[i]);
      bags += offsets[i].numel() - 1;
      total += std::max(ids[i].numel(), offsets[i].numel() - 1);
    }
    const Tensor whole = new_rows({bags, g.dim}, ids[g.members[0]]);
    float* base = whole.mutable_data_ptr<float>();
    int64_t at = 0;
    for (size_t m = 0; m < g.members.size(); ++m) {
      const int i = g.members[m];
      const int64_t mine = offsets[i].numel() - 1;
      outs[i] = piece_of(whole, at, {mine, g.dim});
      parts[m] = krk_pooled_part{id_ptr(ids[i]), ids[i].numel(), off_ptr(offsets[i]), mine, float_ptr(weights[i]),
                                 base + at, g.dim, modes[i], (float)patches[i]};
      at += mine * g.dim;
    }
    krk_group* h = g.h->get();
    KRK_CALL(krk_group_set_stream, h, stream);
    const int32_t rc =
        total > c->combined_max
            ? KRK_E_CAPACITY
            : krk_group_pull_pooled_parts(h, parts.data(), kFlags | (record ? KRK_NOTE_ROWS : 0u));
    if (rc == KRK_SUCCESS) continue;
    if (rc != KRK_E_CAPACITY) fail(rc, "krk_group_pull_pooled_parts");
    combined = false;
    for (size_t m = 0; m < g.members.size(); ++m) {
      const krk_pooled_part& p = parts[m];
      KRK_CALL(krk_sparse_pull_pooled, c->tables[g.members[m]]->get(), p.ids, p.n, p.offsets, p.bags, p.weights,
               p.mode, p.patch_value, p.rows, kFlags);
    }
  }
  if (record) {
    auto node = new_node<CombineJaggedBackward>(param);
    node->c = c;
    node->combined = combined;
    node->modes = modes;
    for (const Tensor& t : ids) node->ids.emplace_back(t, false);
    for (const Tensor& t : offsets) node->offsets.emplace_back(t, false);
    node->weights = weights;
    for (Tensor& o : outs) torch::autograd::set_history(o, node);
  }
  return outs;
}

}  // namespace

// Handles and optimizers come as the ctypes objects that hold them (see Bound).
PYBIND11_MODULE(_torch_native, m) {
  using release = py::call_guard<py::gil_scoped_release>;
  py::class_<Table, TablePtr>(m, "Table")
      .def(py::init([](const py::object& h, const py::object& optim, int64_t dim, double lr) {
        return std::shared_ptr<Table>(new Table{Bound<krk_sparse*>(h), Bound<krk_optim>(optim), dim, lr});
      }))
      .def("bind_table", [](Table& t, const py::object& h) { t.h.bind(h); })
      .def("bind_optim", [](Table& t, const py::object& optim) { t.optim.bind(optim); })
      .def_readwrite("lr", &Table::lr);
  py::class_<Combine, CombinePtr>(m, "Combine")
      .def(py::init([](const std::vector<std::tuple<py::object, int64_t, std::vector<int>>>& groups,
                       const std::vector<py::object>& tables, const std::vector<int64_t>& dims,
                       const py::object& optim, double lr) {
        std::shared_ptr<Combine> c(new Combine{{}, {}, dims, Bound<krk_optim>(optim), lr});
        for (const auto& [h, dim, members] : groups)
          c->groups.push_back({std::make_unique<Bound<krk_group*>>(h), dim, members});
        for (const py::object& t : tables) c->tables.push_back(std::make_unique<Bound<krk_sparse*>>(t));
        return c;
      }))
      .def("bind_optim", [](Combine& c, const py::object& optim) { c.optim.bind(optim); })
      .def_readwrite("lr", &Combine::lr)
      .def_readwrite("combined_max", &Combine::combined_max);
  m.def("embedding", &embedding, release());
  m.def("jagged", &jagged, release());
  m.def("combine", &combine, release());
  m.def("combine_jagged", &combine_jagged, release());
}

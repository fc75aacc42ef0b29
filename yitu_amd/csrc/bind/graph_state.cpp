// State derived from a graph's index tensors: the widest row, the row plan, the by-source
// view. An entry belongs to a tensor OBJECT (its implementation's address, which a weak
// reference keeps from being reused), at one data address and version; Python builds the
// entries on a miss (yitu_amd/_lib.py, yitu_amd/graph_ext.py), stores them here and drops
// them when the tensor dies or is named to forget(). A use on another stream than the one
// an entry was built on waits for the build's event (_lib._Built).
#include <memory>
#include <mutex>

#include "bind.hpp"

namespace yitu_bind {
namespace {

struct Owner {
    c10::weak_intrusive_ptr<c10::TensorImpl> ref;
    const void *data;
    int64_t numel;
    uint32_t version;
    explicit Owner(const Tensor &t)
        : ref(t.getIntrusivePtr()), data(t.const_data_ptr()), numel(t.numel()),
          version(t._version()) {}
    bool is(const Tensor &t) const {
        return data == t.const_data_ptr() && numel == t.numel() && version == t._version();
    }
};

struct Key {
    const void *a, *b;
    int64_t n_src;
    int mask;
    bool operator==(const Key &o) const {
        return a == o.a && b == o.b && n_src == o.n_src && mask == o.mask;
    }
};
struct KeyHash {
    size_t operator()(const Key &k) const {
        size_t h = reinterpret_cast<size_t>(k.a) * 0x9E3779B97F4A7C15ull;
        h ^= reinterpret_cast<size_t>(k.b) * 0xC2B2AE3D27D4EB4Full + (h >> 29);
        return h ^ ((size_t)k.n_src * 0x165667B19E3779F9ull + (size_t)k.mask);
    }
};
struct Degree {
    Owner indptr;
    int64_t value;
};
// A Python object that threads without the interpreter lock may take and give back.
struct Held {
    py::object object;
    explicit Held(py::object o) : object(std::move(o)) {}
    ~Held() {
        py::gil_scoped_acquire gil;
        object = py::object();
    }
};
using HeldPtr = std::shared_ptr<Held>;
struct Built {
    Owner indptr, indices;
    HeldPtr built;     // _lib._Built
    py::object value;  // the plan tensor, or graph_ext's by-source object
    void *stream;
    BySource view;  // by-source entries only
    OptTensor plan;
};

struct Weights {  // edge weights that came by, and their copy in by-source order
    Owner values, indptr, indices;
    int64_t n_src;
    OptTensor copy;
    HeldPtr built;  // _lib._Built of the copy
    void *stream;
};

std::mutex lock;
// (never destroyed: at the end of the process the interpreter is gone before these are)
using BuiltMap = std::unordered_map<Key, Built, KeyHash>;
auto &degrees = *new std::unordered_map<const void *, Degree>;
auto &plans = *new BuiltMap;
auto &views = *new BuiltMap;
auto &weights = *new std::unordered_map<const void *, Weights>;

const void *id(const Tensor &t) { return t.unsafeGetTensorImpl(); }
void *stream_of(const Tensor &t) {
    return t.is_cuda() ? c10::hip::getCurrentHIPStream(t.device().index()).stream() : nullptr;
}

int64_t find_degree(const Tensor &indptr) {
    std::lock_guard<std::mutex> g(lock);
    auto it = degrees.find(id(indptr));
    return it != degrees.end() && it->second.indptr.is(indptr) ? it->second.value : -1;
}

// Calls found(entry) under the lock; false when there is no entry. *wait is set when the
// caller has to wait for the entry's event (with the interpreter lock, after this returns):
// a reference of its own, another thread may drop the entry meanwhile.
template <typename F>
bool find_built(BuiltMap &map, const Tensor &indptr,
                const Tensor &indices, int64_t n_src, int mask, HeldPtr *wait, F found) {
    std::lock_guard<std::mutex> g(lock);
    auto it = map.find(Key{id(indices), id(indptr), n_src, mask});
    if (it == map.end() || !it->second.indices.is(indices) || !it->second.indptr.is(indptr))
        return false;
    *wait = it->second.stream != stream_of(indices) ? it->second.built : nullptr;
    found(it->second);
    return true;
}
void wait_for(const HeldPtr &built, const Tensor &t) {
    if (!built) return;
    py::gil_scoped_acquire gil;
    built->object.attr("get")(py::cast(t.device()));
}

int64_t max_degree(const Tensor &indptr) {
    const int64_t v = find_degree(indptr);
    if (v >= 0) return v;
    py::gil_scoped_acquire gil;
    return py::module_::import("yitu_amd._lib").attr("max_degree")(indptr).cast<int64_t>();
}

void put_built(BuiltMap &map, const Tensor &indptr,
               const Tensor &indices, int64_t n_src, int mask, const py::object &built,
               bool view) {
    Built b{Owner(indptr), Owner(indices), std::make_shared<Held>(built), built.attr("value"), stream_of(indices), {}, {}};
    if (view) b.view = by_source_of(b.value);
    else b.plan = b.value.cast<Tensor>();
    std::optional<Built> old;  // destroyed after the lock is given back
    std::lock_guard<std::mutex> g(lock);
    const Key key{id(indices), id(indptr), n_src, mask};
    auto it = map.find(key);
    if (it != map.end()) {
        old = std::move(it->second);
        map.erase(it);
    }
    map.emplace(key, std::move(b));
}

void drop(const void *impl) {
    std::vector<Built> old;  // destroyed after the lock is given back
    std::vector<Weights> old_weights;
    {
        std::lock_guard<std::mutex> g(lock);
        degrees.erase(impl);
        for (auto it = weights.begin(); it != weights.end();)
            if (it->first == impl || it->second.indptr.ref._unsafe_get_target() == impl ||
                it->second.indices.ref._unsafe_get_target() == impl) {
                old_weights.push_back(std::move(it->second));
                it = weights.erase(it);
            } else
                ++it;
        for (auto *map : {&plans, &views})
            for (auto it = map->begin(); it != map->end();)
                if (it->first.a == impl || it->first.b == impl) {
                    old.push_back(std::move(it->second));
                    it = map->erase(it);
                } else
                    ++it;
    }
}

}  // namespace

BySource by_source_of(const py::handle &t) {
    BySource b;
    b.t_indptr = t.attr("t_indptr").cast<Tensor>();
    b.t_rows = t.attr("t_rows").cast<Tensor>();
    b.t_perm = t.attr("t_perm").cast<Tensor>();
    b.max_degree = t.attr("max_degree_t").cast<int64_t>();
    b.plan = t.attr("plan_t").cast<OptTensor>();
    return b;
}

RowState row_state(const Tensor &indptr, const Tensor &indices, int64_t n_src, int mask) {
    RowState s;
    s.max_degree = max_degree(indptr);
    // as _lib.row_plan: no plan for small graphs without long rows
    if (s.max_degree < kLongRow && indices.numel() < kPlanMinEdges) return s;
    HeldPtr wait;
    if (find_built(plans, indptr, indices, n_src, mask, &wait, [&](Built &b) { s.plan = b.plan; })) {
        wait_for(wait, indices);
        return s;
    }
    py::gil_scoped_acquire gil;
    s.plan = py::module_::import("yitu_amd._lib")
                 .attr("row_plan")(indptr, indices, n_src, mask)
                 .cast<OptTensor>();
    return s;
}

BySource by_source(const Tensor &indptr, const Tensor &indices, int64_t n_src) {
    BySource s;
    HeldPtr wait;
    if (find_built(views, indptr, indices, n_src, 0, &wait, [&](Built &b) { s = b.view; })) {
        wait_for(wait, indices);
        return s;
    }
    py::gil_scoped_acquire gil;
    return by_source_of(
        py::module_::import("yitu_amd.graph_ext").attr("transposed")(indptr, indices, n_src));
}

// Whether the stream of a call on `t` records a graph.
static bool recording(const Tensor &t) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    C10_HIP_CHECK(hipStreamIsCapturing(static_cast<hipStream_t>(stream_of(t)), &status));
    return status != hipStreamCaptureStatusNone;
}

// Edge weights that take no gradient are usually constants of the graph (norms), passed
// again every step. The backward reads them through the edge permutation, a scattered
// 4-byte read per edge and head; the second time the same tensor (same version) comes by a
// copy in by-source order is made and kept for as long as the tensor lives (`force`: at
// once). Nothing is returned the first time. While the stream records a graph none is kept: its
// memory would hold the weights only from the first replay on.
OptTensor by_source_values(const Tensor &values, const Tensor &indptr, const Tensor &indices,
                           int64_t n_src, bool force) {
    bool known = false, seen = false;
    OptTensor copy;
    HeldPtr wait;
    {
        std::lock_guard<std::mutex> g(lock);
        auto it = weights.find(id(values));
        known = it != weights.end();
        seen = known && it->second.values.is(values) && it->second.n_src == n_src &&
               it->second.indptr.ref._unsafe_get_target() == id(indptr) &&
               it->second.indices.ref._unsafe_get_target() == id(indices) &&
               it->second.indptr.is(indptr) && it->second.indices.is(indices);
        if (seen && it->second.copy) {
            copy = it->second.copy;
            if (it->second.stream != stream_of(values)) wait = it->second.built;
        }
    }
    if (copy) {
        wait_for(wait, values);
        return copy;
    }
    if (recording(values)) {
        if (force) copy = values.index_select(0, by_source(indptr, indices, n_src).t_perm);
        return copy;
    }
    if (!known) {
        py::gil_scoped_acquire gil;
        py::module_::import("yitu_amd._lib").attr("watch")(values);
    }
    HeldPtr built;
    if (seen || force) {
        copy = values.index_select(0, by_source(indptr, indices, n_src).t_perm);
        py::gil_scoped_acquire gil;
        built = std::make_shared<Held>(
            py::module_::import("yitu_amd._lib").attr("_Built")(*copy, py::cast(values.device())));
    }
    std::optional<Weights> old;  // destroyed after the lock is given back
    std::lock_guard<std::mutex> g(lock);
    auto it = weights.find(id(values));
    if (it != weights.end()) {
        old = std::move(it->second);
        weights.erase(it);
    }
    weights.emplace(id(values), Weights{Owner(values), Owner(indptr), Owner(indices), n_src, copy,
                                        built, stream_of(values)});
    return copy;
}

void bind_graph_state(py::module_ &m) {
    m.def("by_source_values", &by_source_values);
    m.def("find_max_degree", &find_degree);
    m.def("put_max_degree", [](const Tensor &indptr, int64_t v) {
        std::lock_guard<std::mutex> g(lock);
        degrees.insert_or_assign(id(indptr), Degree{Owner(indptr), v});
    });
    const auto find = [](auto &map, const Tensor &indptr, const Tensor &indices, int64_t n_src,
                         int mask) -> py::object {
        py::object value = py::none();
        HeldPtr wait;
        if (find_built(map, indptr, indices, n_src, mask, &wait, [&](Built &b) { value = b.value; }))
            wait_for(wait, indices);
        return value;
    };
    m.def("find_plan", [find](const Tensor &indptr, const Tensor &indices, int64_t n_src, int mask) {
        return find(plans, indptr, indices, n_src, mask);
    });
    m.def("find_by_source", [find](const Tensor &indptr, const Tensor &indices, int64_t n_src) {
        return find(views, indptr, indices, n_src, 0);
    });
    m.def("put_plan", [](const Tensor &indptr, const Tensor &indices, int64_t n_src, int mask,
                         const py::object &built) {
        put_built(plans, indptr, indices, n_src, mask, built, false);
    });
    m.def("put_by_source", [](const Tensor &indptr, const Tensor &indices, int64_t n_src,
                              const py::object &built) {
        put_built(views, indptr, indices, n_src, 0, built, true);
    });
    // identity, address and version of every tensor, as one comparable value
    m.def("tensor_state", [](const TensorVec &ts) {
        std::vector<uintptr_t> v;
        v.reserve(3 * ts.size());
        for (const Tensor &t : ts) {
            v.push_back(reinterpret_cast<uintptr_t>(id(t)));
            v.push_back(reinterpret_cast<uintptr_t>(t.const_data_ptr()));
            v.push_back(t._version());
        }
        return py::bytes(reinterpret_cast<const char *>(v.data()), v.size() * sizeof(v[0]));
    });
    m.def("impl_of", [](const Tensor &t) { return reinterpret_cast<uintptr_t>(id(t)); });
    m.def("drop", [](uintptr_t impl) { drop(reinterpret_cast<const void *>(impl)); });
}

}  // namespace yitu_bind

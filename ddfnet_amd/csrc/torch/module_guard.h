// Cheap answer to "are these Python modules still what they were when a plan was made of
// them?".  A plan (the tensors and constants of a module tree, collected once in Python)
// stays valid while
//   - every module has its class, its attributes the plan was made from, and its own
//     dictionaries of parameters, buffers and sub-modules, and those hold the same entries
//     in the same order (nothing replaced, added or taken out);
//   - no attribute of a module hides something of its class or tables (an instance's
//     `forward`, a tensor assigned over a parameter);
//   - the methods of the classes that the plan stands for are the ones this package knows;
//   - nobody listens on a module (hooks).
// Asking that through the interpreter on every call costs more than launching a layer's
// kernels.  CPython up to 3.11 stamps a dictionary anew with every change (PEP 509): as long
// as the stamps are the ones seen last nothing has changed, and only dictionaries with
// another stamp are looked through.  Without stamps all of them are, on every call.
// In-place changes of a parameter (optimizer steps, load_state_dict, .half(), .to()) keep
// the object and are seen by whoever reads the tensor.
#pragma once

#include <torch/extension.h>

#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <memory>
#include <unordered_set>
#include <vector>

namespace ddf_torch {

namespace py = pybind11;

#if PY_VERSION_HEX < 0x030C0000
constexpr bool kDictStamps = true;
inline uint64_t stamp_of(PyObject *dict) { return reinterpret_cast<PyDictObject *>(dict)->ma_version_tag; }
#else
constexpr bool kDictStamps = false;
inline uint64_t stamp_of(PyObject *) { return 0; }
#endif

// Python objects that something native owns, known to the cycle collector by `traverse` and
// `clear` (see collectable): a module tree may lead back to whoever holds on to it.
class Refs {
public:
    Refs() = default;
    Refs(const Refs &) = delete;
    Refs &operator=(const Refs &) = delete;
    ~Refs() { clear(); }
    PyObject *add(PyObject *o) {
        Py_XINCREF(o);
        if (o) objects_.push_back(o);
        return o;
    }
    int traverse(visitproc visit, void *arg) const {
        for (PyObject *o : objects_) Py_VISIT(o);
        return 0;
    }
    void clear() {
        std::vector<PyObject *> gone;
        gone.swap(objects_);
        for (PyObject *o : gone) Py_DECREF(o);
    }

private:
    std::vector<PyObject *> objects_;
};

// pybind11::custom_type_setup of a class whose `traverse` and `clear` are those of its Refs.
template <class T>
void collectable(PyHeapTypeObject *heap_type) {
    PyTypeObject *type = &heap_type->ht_type;
    type->tp_flags |= Py_TPFLAGS_HAVE_GC;
    type->tp_traverse = [](PyObject *self, visitproc visit, void *arg) -> int {
        Py_VISIT(Py_TYPE(self));
        auto at = reinterpret_cast<py::detail::instance *>(self)->get_value_and_holder();
        return at.holder_constructed() ? static_cast<const T *>(at.value_ptr())->traverse(visit, arg) : 0;
    };
    type->tp_clear = [](PyObject *self) -> int {
        auto at = reinterpret_cast<py::detail::instance *>(self)->get_value_and_holder();
        if (at.holder_constructed()) static_cast<T *>(at.value_ptr())->clear();
        return 0;
    };
}

// A tensor by its Python object (that some Refs owns; null: none).  The collector sees through
// an owned Python object, which it does not through an at::Tensor.
class TensorRef {
public:
    TensorRef() = default;
    explicit TensorRef(PyObject *o) : o_(o) {
        TORCH_CHECK(!o || THPVariable_Check(o), "tensors expected");
    }
    bool defined() const { return o_ != nullptr; }
    const at::Tensor &operator*() const { return THPVariable_Unpack(o_); }
    const at::Tensor *operator->() const { return &THPVariable_Unpack(o_); }

private:
    PyObject *o_ = nullptr;
};
// The objects of a list, owned by `refs`; None: no tensor.
inline std::vector<TensorRef> tensor_refs(Refs &refs, const py::list &objects) {
    std::vector<TensorRef> out;
    for (auto o : objects) out.emplace_back(o.is_none() ? nullptr : refs.add(o.ptr()));
    return out;
}
inline const void *ptr_or_null(const TensorRef &t) { return t.defined() ? t->data_ptr() : nullptr; }

inline std::vector<PyObject *> interned(std::initializer_list<const char *> names) {
    std::vector<PyObject *> out;
    for (const char *name : names) out.push_back(PyUnicode_InternFromString(name));
    return out;
}

// Of the module a plan is made for the guard keeps no more than a weak reference: the plan hangs
// on that module, and a model goes with its last user, not at some later collection.
class ModuleGuard {
public:
    // What is fixed for the package, collected once (modules.py):
    //   classes    {class: (attribute names, ((method name, function), ...))}; a subclass goes
    //              by its nearest ancestor listed, a module of any other class has no guard
    //   own        {class: method names} of the module a plan belongs to: its other methods are
    //              on the way to the plan and may be wrapped, and its own hooks run around it
    //   operators  ((dictionary, key, object), ...) that must be found as they are
    //   silent     dictionaries that must stay empty
    struct Rules {
        py::dict classes, own;
        py::tuple operators, silent;
    };

    // A guard of `modules` (the first is the plan's owner), or null where they are not plain
    // modules of the classes known, or somebody listens.
    static std::unique_ptr<ModuleGuard> make(const Rules &rules, const py::list &modules) {
        std::unique_ptr<ModuleGuard> g(new ModuleGuard());
        for (auto item : rules.operators) {
            PyObject *t = g->keep_.add(item.ptr());
            g->operators_.push_back({PyTuple_GetItem(t, 0), PyTuple_GetItem(t, 1), PyTuple_GetItem(t, 2)});
        }
        for (auto d : rules.silent) g->add_silent(d.ptr());
        bool first = true;
        for (auto m : modules) {
            if (!g->add_module(rules, m.ptr(), first)) return nullptr;
            first = false;
        }
        if (!g->holds()) g.reset();
        return g;
    }

    // Every one of the tensors is an entry of a module's tables or an attribute relied on (a
    // tensor assigned as a plain attribute, as on the replicas of nn.DataParallel, is not: the
    // guard does not see it replaced), and none is the result of other operations: a plan that
    // holds it would hold its graph (the weights torch.func.functional_call puts in for one call).
    bool covers(const py::list &tensors) const {
        std::unordered_set<PyObject *> mine;
        for (const Pair &p : pairs_) mine.insert(p.value);
        return std::all_of(tensors.begin(), tensors.end(), [&](py::handle o) {
            return o.is_none() || (mine.count(o.ptr()) && THPVariable_Check(o.ptr()) && THPVariable_Unpack(o.ptr()).is_leaf());
        });
    }
    // (caller holds the GIL)
    bool holds() const {
        PyObject *owner = owner_ ? PyWeakref_GetObject(owner_) : Py_None;
        if (owner == Py_None || Py_TYPE(owner) != owner_type_) return false;
        PyObject **attributes = _PyObject_GetDictPtr(owner);
        if (!attributes || *attributes != owner_attributes_) return false;
        for (const Entry &e : operators_)
            if (PyDict_GetItem(e.dict, e.key) != e.value) return false;
        for (PyObject *d : silent_)
            if (PyDict_GET_SIZE(d) != 0) return false;
        for (const Typed &t : modules_)
            if (Py_TYPE(t.module) != t.type) return false;
        for (const Watch &w : watches_) {
            const uint64_t now = stamp_of(w.dict);
            if (kDictStamps && now == w.stamp) continue;
            if (!same(w)) return false;
            w.stamp = now;
        }
        return true;
    }

    int traverse(visitproc visit, void *arg) const { return keep_.traverse(visit, arg); }
    void clear() {
        owner_ = nullptr;     // (never holds again)
        keep_.clear();
    }

private:
    enum Kind { kTable, kAttributes, kClass };
    struct Entry { PyObject *dict, *key, *value; };
    struct Typed { PyObject *module; PyTypeObject *type; };
    struct Watch {
        PyObject *dict;
        Kind kind;
        int first, count;            // kTable: pairs_ of its entries; kAttributes: of those relied on
        PyTypeObject *type = nullptr;   // kAttributes: the module's class
        PyObject *tables[3] = {nullptr, nullptr, nullptr};
        PyObject *hiding = nullptr;  // kAttributes of the owner: methods not to be hidden (else: any)
        mutable uint64_t stamp;
    };
    struct Pair { PyObject *key, *value; };
    struct Method { PyTypeObject *type; PyObject *name, *value; };

    ModuleGuard() = default;

    void add_silent(PyObject *d) {
        keep_.add(d);
        silent_.push_back(d);
    }
    bool add_module(const Rules &rules, PyObject *m, bool owner) {
        PyTypeObject *type = Py_TYPE(m);
        PyObject *rule = nullptr, *mro = type->tp_mro;
        for (Py_ssize_t i = 0; !rule && i < PyTuple_GET_SIZE(mro); ++i)
            rule = PyDict_GetItem(rules.classes.ptr(), PyTuple_GET_ITEM(mro, i));
        PyObject **slot = _PyObject_GetDictPtr(m);
        if (!rule || !PyTuple_Check(rule) || !slot || !*slot) return false;
        PyObject *attributes = *slot;
        PyObject *own = nullptr;
        for (Py_ssize_t i = 0; owner && !own && i < PyTuple_GET_SIZE(mro); ++i)
            own = PyDict_GetItem(rules.own.ptr(), PyTuple_GET_ITEM(mro, i));
        if (owner && !own) return false;
        if (owner) {
            py::object ref = py::reinterpret_steal<py::object>(PyWeakref_NewRef(m, nullptr));
            if (!ref) throw py::error_already_set();
            owner_ = keep_.add(ref.ptr());
            owner_type_ = type;
            owner_attributes_ = attributes;
        } else {
            keep_.add(m);
            keep_.add(attributes);
            modules_.push_back({m, type});
        }
        if (!add_class(type, PyTuple_GET_ITEM(rule, 1), own)) return false;

        Watch w;
        w.dict = attributes;
        w.kind = kAttributes;
        w.type = type;
        w.hiding = own;
        w.first = (int)pairs_.size();
        auto rely_on = [&](PyObject *key) {
            PyObject *value = PyDict_GetItem(attributes, key);
            if (value) add_pair(key, value);
            return value;
        };
        PyObject *names = PyTuple_GET_ITEM(rule, 0);
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(names); ++i) rely_on(PyTuple_GET_ITEM(names, i));
        for (int i = 0; i < 3; ++i) {
            PyObject *table = rely_on(table_names()[i]);
            // (an ordered dictionary keeps an order of its own)
            if (!table || !PyDict_CheckExact(table)) return false;
            w.tables[i] = table;
        }
        if (!owner)
            for (PyObject *name : hook_names()) {
                PyObject *hooks = rely_on(name);
                if (!hooks) continue;
                if (!PyDict_Check(hooks)) return false;
                add_silent(hooks);
            }
        w.count = (int)pairs_.size() - w.first;
        if (hides(w)) return false;
        w.stamp = stamp_of(attributes);
        watches_.push_back(w);

        for (PyObject *table : w.tables) {
            Watch t;
            t.dict = table;
            t.kind = kTable;
            t.first = (int)pairs_.size();
            Py_ssize_t pos = 0;
            PyObject *key, *value;
            while (PyDict_Next(table, &pos, &key, &value)) add_pair(key, value);
            t.count = (int)pairs_.size() - t.first;
            t.stamp = stamp_of(table);
            watches_.push_back(t);
        }
        return true;
    }
    // The class's methods are the known ones (of a plan's owner: those in `own`).
    bool add_class(PyTypeObject *type, PyObject *methods, PyObject *own) {
        if (std::find(classes_.begin(), classes_.end(), type) != classes_.end()) return true;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(methods); ++i) {
            PyObject *pair = PyTuple_GET_ITEM(methods, i), *name = PyTuple_GET_ITEM(pair, 0);
            if (own && PySequence_Contains(own, name) != 1) continue;
            keep_.add(pair);
            methods_.push_back({type, name, PyTuple_GET_ITEM(pair, 1)});
            if (!as_known(methods_.back())) return false;
        }
        if (!own) classes_.push_back(type);   // (the owner's class may come again below it)
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(type->tp_mro); ++i) {
            PyTypeObject *t = reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(type->tp_mro, i));
            if (t == &PyBaseObject_Type || !t->tp_dict) continue;
            const auto seen = [&](const Watch &w) { return w.dict == t->tp_dict; };
            if (std::any_of(watches_.begin(), watches_.end(), seen)) continue;
            keep_.add(reinterpret_cast<PyObject *>(t));
            Watch w;
            w.dict = t->tp_dict;
            w.kind = kClass;
            w.first = w.count = 0;
            w.stamp = stamp_of(w.dict);
            watches_.push_back(w);
        }
        return true;
    }
    void add_pair(PyObject *key, PyObject *value) {
        keep_.add(key);
        keep_.add(value);
        pairs_.push_back({key, value});
    }

    static bool as_known(const Method &m) {
        return _PyType_Lookup(m.type, m.name) == m.value;
    }
    // An attribute by which the module is not the one its class and tables describe.
    static bool hides(const Watch &w) {
        PyObject *key, *value;
        for (PyObject *table : w.tables)
            for (Py_ssize_t pos = 0; PyDict_Next(table, &pos, &key, &value);)
                if (PyDict_Contains(w.dict, key) != 0) return true;
        if (w.hiding) {
            for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(w.hiding); ++i)
                if (PyDict_Contains(w.dict, PyTuple_GET_ITEM(w.hiding, i)) != 0) return true;
            return false;
        }
        for (Py_ssize_t pos = 0; PyDict_Next(w.dict, &pos, &key, &value);)
            if (_PyType_Lookup(w.type, key)) return true;
        return false;
    }
    bool same(const Watch &w) const {
        if (w.kind == kClass) return std::all_of(methods_.begin(), methods_.end(), as_known);
        const Pair *p = pairs_.data() + w.first;
        PyObject *key, *value;
        Py_ssize_t pos = 0;
        if (w.kind == kTable) {
            if (PyDict_GET_SIZE(w.dict) != w.count) return false;
            for (int i = 0; PyDict_Next(w.dict, &pos, &key, &value); ++i)
                if (value != p[i].value || (key != p[i].key && PyObject_RichCompareBool(key, p[i].key, Py_EQ) != 1))
                    return false;
            return true;
        }
        for (int i = 0; i < w.count; ++i)
            if (PyDict_GetItem(w.dict, p[i].key) != p[i].value) return false;
        return !hides(w);
    }

    static const std::vector<PyObject *> &table_names() {
        static const auto *names = new std::vector<PyObject *>(interned({"_modules", "_parameters", "_buffers"}));
        return *names;
    }
    static const std::vector<PyObject *> &hook_names() {
        static const auto *names = new std::vector<PyObject *>(
            interned({"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"}));
        return *names;
    }

    Refs keep_;                        // owns what is below, but for the owner's attributes
    PyObject *owner_ = nullptr;        // weak reference
    PyTypeObject *owner_type_ = nullptr;
    PyObject *owner_attributes_ = nullptr;
    std::vector<Entry> operators_;
    std::vector<PyObject *> silent_;
    std::vector<Typed> modules_;
    std::vector<PyTypeObject *> classes_;
    std::vector<Method> methods_;
    std::vector<Pair> pairs_;
    std::vector<Watch> watches_;
};

// Nothing at all about a tree of modules (the first is its root, held weakly as above) has
// changed: their classes, attributes, tables, hooks, the operators.  What was found wanting then
// is still: a network that is not stock is looked through once and not on every call.
class ModuleSnapshot {
public:
    ModuleSnapshot(const ModuleGuard::Rules &rules, const py::list &modules) {
        static const auto *names = new std::vector<PyObject *>(
            interned({"_modules", "_parameters", "_buffers", "_forward_hooks", "_forward_pre_hooks", "_backward_hooks",
                      "_backward_pre_hooks"}));
        for (auto item : rules.operators) {
            PyObject *t = keep_.add(item.ptr()), *dict = PyTuple_GetItem(t, 0), *key = PyTuple_GetItem(t, 1);
            operators_.push_back({dict, key, keep_.add(PyDict_GetItem(dict, key))});
        }
        for (auto d : rules.silent) watch(keep_.add(d.ptr()));
        std::unordered_set<PyObject *> classes;
        for (auto item : modules) {
            PyObject *m = item.ptr(), **slot = _PyObject_GetDictPtr(m);
            if (!slot || !*slot || !kDictStamps) return;    // (never holds)
            const bool root = owner_ == nullptr;
            if (root) {
                py::object ref = py::reinterpret_steal<py::object>(PyWeakref_NewRef(m, nullptr));
                if (!ref) throw py::error_already_set();
                owner_ = keep_.add(ref.ptr());
                owner_type_ = Py_TYPE(m);
                owner_attributes_ = *slot;
            } else {
                modules_.emplace_back(keep_.add(m), Py_TYPE(m));
                keep_.add(*slot);
            }
            watch(*slot);
            for (PyObject *name : *names) {
                PyObject *d = PyDict_GetItem(*slot, name);
                if (d && PyDict_Check(d)) watch(keep_.add(d));
            }
            PyObject *mro = Py_TYPE(m)->tp_mro;
            for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(mro); ++i) {
                PyTypeObject *t = reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(mro, i));
                if (t == &PyBaseObject_Type || !t->tp_dict || !classes.insert((PyObject *)t).second) continue;
                keep_.add(reinterpret_cast<PyObject *>(t));
                watch(t->tp_dict);
            }
        }
        whole_ = true;
    }
    // (caller holds the GIL)
    bool holds() const {
        PyObject *owner = whole_ && owner_ ? PyWeakref_GetObject(owner_) : Py_None;
        if (owner == Py_None || Py_TYPE(owner) != owner_type_) return false;
        PyObject **attributes = _PyObject_GetDictPtr(owner);
        if (!attributes || *attributes != owner_attributes_) return false;
        for (const auto &e : operators_)
            if (PyDict_GetItem(e.dict, e.key) != e.value) return false;
        for (const auto &m : modules_)
            if (Py_TYPE(m.first) != m.second) return false;
        for (const auto &w : watches_)
            if (stamp_of(w.first) != w.second) return false;
        return true;
    }
    int traverse(visitproc visit, void *arg) const { return keep_.traverse(visit, arg); }
    void clear() {
        whole_ = false;
        owner_ = nullptr;
        keep_.clear();
    }

private:
    struct Entry { PyObject *dict, *key, *value; };
    void watch(PyObject *dict) { watches_.emplace_back(dict, stamp_of(dict)); }

    Refs keep_;                        // owns what is below, but for the root's attributes
    bool whole_ = false;
    PyObject *owner_ = nullptr, *owner_attributes_ = nullptr;
    PyTypeObject *owner_type_ = nullptr;
    std::vector<Entry> operators_;
    std::vector<std::pair<PyObject *, PyTypeObject *>> modules_;
    std::vector<std::pair<PyObject *, uint64_t>> watches_;
};

}  // namespace ddf_torch

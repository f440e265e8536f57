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
    static std::shared_ptr<ModuleGuard> make(const Rules &rules, const py::list &modules) {
        std::shared_ptr<ModuleGuard> g(new ModuleGuard());
        for (auto item : rules.operators) {
            py::tuple t = py::reinterpret_borrow<py::tuple>(item);
            g->keep_.append(t);
            g->operators_.push_back({t[0].ptr(), t[1].ptr(), t[2].ptr()});
        }
        for (auto d : rules.silent) g->add_silent(d.ptr());
        bool first = true;
        for (auto m : modules) {
            if (!g->add_module(rules, m.ptr(), first)) return nullptr;
            first = false;
        }
        return g->holds() ? g : nullptr;
    }

    // Every one of the objects is an entry of a module's tables or an attribute relied on (a
    // tensor assigned as a plain attribute, as on the replicas of nn.DataParallel, is not: the
    // guard does not see it replaced).
    bool covers(const py::list &objects) const {
        std::unordered_set<PyObject *> mine;
        for (const Pair &p : pairs_) mine.insert(p.value);
        return std::all_of(objects.begin(), objects.end(),
                           [&](py::handle o) { return o.is_none() || mine.count(o.ptr()); });
    }
    // (caller holds the GIL)
    bool holds() const {
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

private:
    enum Kind { kTable, kAttributes, kClass };
    struct Entry { PyObject *dict, *key, *value; };
    struct Typed { PyObject *module; PyTypeObject *type; };
    struct Watch {
        PyObject *dict;
        Kind kind;
        int first, count;            // kTable: pairs_ of its entries; kAttributes: of those relied on
        int module = 0;              // kAttributes: index into modules_
        PyObject *tables[3] = {nullptr, nullptr, nullptr};
        PyObject *hiding = nullptr;  // kAttributes of the owner: methods not to be hidden (else: any)
        mutable uint64_t stamp;
    };
    struct Pair { PyObject *key, *value; };
    struct Method { PyTypeObject *type; PyObject *name, *value; };

    ModuleGuard() = default;

    void add_silent(PyObject *d) {
        keep_.append(py::reinterpret_borrow<py::object>(d));
        silent_.push_back(d);
    }
    bool add_module(const Rules &rules, PyObject *m, bool owner) {
        PyTypeObject *type = Py_TYPE(m);
        PyObject *rule = nullptr, *mro = type->tp_mro;
        for (Py_ssize_t i = 0; !rule && i < PyTuple_GET_SIZE(mro); ++i)
            rule = PyDict_GetItem(rules.classes.ptr(), PyTuple_GET_ITEM(mro, i));
        PyObject **slot = _PyObject_GetDictPtr(m);
        if (!rule || !slot || !*slot) return false;
        PyObject *attributes = *slot;
        PyObject *own = nullptr;
        for (Py_ssize_t i = 0; owner && !own && i < PyTuple_GET_SIZE(mro); ++i)
            own = PyDict_GetItem(rules.own.ptr(), PyTuple_GET_ITEM(mro, i));
        if (owner && !own) return false;
        keep_.append(py::reinterpret_borrow<py::object>(m));
        keep_.append(py::reinterpret_borrow<py::object>(attributes));
        modules_.push_back({m, type});
        if (!add_class(type, PyTuple_GET_ITEM(rule, 1), own)) return false;

        Watch w;
        w.dict = attributes;
        w.kind = kAttributes;
        w.module = (int)modules_.size() - 1;
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
            PyObject *table = rely_on(table_names()[i].ptr());
            // (an ordered dictionary keeps an order of its own)
            if (!table || !PyDict_CheckExact(table)) return false;
            w.tables[i] = table;
        }
        if (!owner)
            for (const py::str &name : hook_names()) {
                PyObject *hooks = rely_on(name.ptr());
                if (!hooks) continue;
                if (!PyDict_Check(hooks)) return false;
                add_silent(hooks);
            }
        w.count = (int)pairs_.size() - w.first;
        Py_ssize_t pos = 0;
        PyObject *key, *value;
        while (PyDict_Next(attributes, &pos, &key, &value))
            if (hides(w, key)) return false;
        w.stamp = stamp_of(attributes);
        watches_.push_back(w);

        for (PyObject *table : w.tables) {
            Watch t;
            t.dict = table;
            t.kind = kTable;
            t.first = (int)pairs_.size();
            pos = 0;
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
            keep_.append(py::reinterpret_borrow<py::object>(pair));
            methods_.push_back({type, name, PyTuple_GET_ITEM(pair, 1)});
            if (!as_known(methods_.back())) return false;
        }
        if (!own) classes_.push_back(type);   // (the owner's class may come again below it)
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(type->tp_mro); ++i) {
            PyTypeObject *t = reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(type->tp_mro, i));
            if (t == &PyBaseObject_Type || !t->tp_dict) continue;
            const auto seen = [&](const Watch &w) { return w.dict == t->tp_dict; };
            if (std::any_of(watches_.begin(), watches_.end(), seen)) continue;
            keep_.append(py::reinterpret_borrow<py::object>(reinterpret_cast<PyObject *>(t)));
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
        keep_.append(py::reinterpret_borrow<py::object>(key));
        keep_.append(py::reinterpret_borrow<py::object>(value));
        pairs_.push_back({key, value});
    }

    static bool as_known(const Method &m) {
        return _PyType_Lookup(m.type, m.name) == m.value;
    }
    // An attribute by which the module is not the one its class and tables describe.
    bool hides(const Watch &w, PyObject *key) const {
        for (PyObject *table : w.tables)
            if (PyDict_Contains(table, key) != 0) return true;
        if (w.hiding) return PySequence_Contains(w.hiding, key) != 0;
        return _PyType_Lookup(modules_[w.module].type, key) != nullptr;
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
        while (PyDict_Next(w.dict, &pos, &key, &value))
            if (hides(w, key)) return false;
        return true;
    }

    static const std::vector<py::str> &table_names() {
        static const auto *names = new std::vector<py::str>{"_modules", "_parameters", "_buffers"};
        return *names;
    }
    static const std::vector<py::str> &hook_names() {
        static const auto *names = new std::vector<py::str>{"_forward_hooks", "_forward_pre_hooks", "_backward_hooks",
                                                            "_backward_pre_hooks"};
        return *names;
    }

    py::list keep_;                    // owns every reference below
    std::vector<Entry> operators_;
    std::vector<PyObject *> silent_;
    std::vector<Typed> modules_;
    std::vector<PyTypeObject *> classes_;
    std::vector<Method> methods_;
    std::vector<Pair> pairs_;
    std::vector<Watch> watches_;
};

}  // namespace ddf_torch

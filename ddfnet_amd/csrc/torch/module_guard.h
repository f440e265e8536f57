// Cheap answer to "are these Python modules still what they were when a plan was made of
// them?".  A plan (the tensors and constants of a module tree, collected once in Python)
// stays valid while every attribute, parameter and sub-module it was made from is the
// same object and nobody has registered a hook.  Asking that through the interpreter on
// every call costs more than launching a layer's kernels; here it is one dictionary
// lookup per object.  In-place changes of a parameter (optimizer steps, load_state_dict,
// .half(), .to()) keep the object and are seen by whoever reads the tensor.
#pragma once

#include <torch/extension.h>

#include <vector>

namespace ddf_torch {

namespace py = pybind11;

class ModuleGuard {
public:
    // same: (dictionary, key, the object it held); empty: dictionaries that held nothing.
    ModuleGuard(py::list same, py::list empty) : same_(std::move(same)), empty_(std::move(empty)) {
        for (auto item : same_) {
            py::tuple t = py::reinterpret_borrow<py::tuple>(item);
            entries_.push_back({PyTuple_GET_ITEM(t.ptr(), 0), PyTuple_GET_ITEM(t.ptr(), 1),
                                PyTuple_GET_ITEM(t.ptr(), 2)});
        }
        for (auto item : empty_) dicts_.push_back(item.ptr());
    }
    // (caller holds the GIL)
    bool holds() const {
        for (const Entry &e : entries_)
            if (PyDict_GetItem(e.dict, e.key) != e.value) return false;
        for (PyObject *d : dicts_)
            if (PyDict_Size(d) != 0) return false;
        return true;
    }

private:
    struct Entry { PyObject *dict, *key, *value; };
    py::list same_, empty_;            // own the references
    std::vector<Entry> entries_;
    std::vector<PyObject *> dicts_;
};

}  // namespace ddf_torch

// What the attention layer and the small model look at before a kernel stands in for modules: that nothing hangs on
// the modules which a call would also run, and that their parameters are what kernels can read by address.  Looked at
// anew for every call; in Python a pass over four layers spent longer on it than on its launches.
#include "module_checks.h"

#include <torch/csrc/Device.h>
#include <torch/csrc/autograd/python_variable.h>

namespace GPT {
namespace {

// The object's own dictionary (borrowed), or null.
PyObject* own_dict(PyObject* o) {
    PyObject** at = _PyObject_GetDictPtr(o);
    return at && *at && PyDict_Check(*at) ? *at : nullptr;
}

struct Names {
    PyObject* hooks[4];
    PyObject *forward, *weight, *bias, *parameters, *buffers, *modules, *rotary, *table, *neox, *rotary_dim, *head_size, *head_dim;
    Names() {
        const char* h[4] = { "_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks" };
        for (int i = 0; i < 4; i++) hooks[i] = PyUnicode_InternFromString(h[i]);
        forward = PyUnicode_InternFromString("forward");
        weight = PyUnicode_InternFromString("weight");
        bias = PyUnicode_InternFromString("bias");
        parameters = PyUnicode_InternFromString("_parameters");
        buffers = PyUnicode_InternFromString("_buffers");
        modules = PyUnicode_InternFromString("_modules");
        rotary = PyUnicode_InternFromString("rotary_emb");
        table = PyUnicode_InternFromString("cos_sin_cache");
        neox = PyUnicode_InternFromString("is_neox_style");
        rotary_dim = PyUnicode_InternFromString("rotary_dim");
        head_size = PyUnicode_InternFromString("head_size");
        head_dim = PyUnicode_InternFromString("head_dim");
    }
};
const Names& names() {
    static const Names* n = new Names;               // (interned strings outlive the interpreter's teardown)
    return *n;
}

// dict[key] (borrowed) or null; an error of the look-up is raised.
PyObject* get(PyObject* dict, PyObject* key) {
    PyObject* v = PyDict_GetItemWithError(dict, key);
    if (!v && PyErr_Occurred()) throw py::error_already_set();
    return v;
}

// m.name, without the detour over Module.__getattr__ where that would find a registered module.
py::object attribute(PyObject* m, PyObject* name) {
    PyObject* own = own_dict(m);
    if (own && !_PyType_Lookup(Py_TYPE(m), name) && !get(own, name)) {
        PyObject *parameters = get(own, names().parameters), *buffers = get(own, names().buffers), *modules = get(own, names().modules);
        if (parameters && buffers && modules && PyDict_CheckExact(parameters) && PyDict_CheckExact(buffers) && PyDict_CheckExact(modules) &&
            !get(parameters, name) && !get(buffers, name)) {
            if (PyObject* child = get(modules, name)) return py::reinterpret_borrow<py::object>(child);
        }
    }
    PyObject* v = PyObject_GetAttr(m, name);
    if (!v) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(v);
}

bool is_bare(PyObject* m, PyObject* cls) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(m)) != cls) return false;
    PyObject* own = own_dict(m);
    if (!own) return false;
    for (PyObject* name : names().hooks) {
        PyObject* hooks = get(own, name);
        if (!hooks) return false;
        const int any = PyObject_IsTrue(hooks);
        if (any < 0) throw py::error_already_set();
        if (any) return false;
    }
    return get(own, names().forward) == nullptr;
}

// device: a torch.device, or what compares itself with one
bool is_on(const at::Tensor& t, py::handle device) {
    if (THPDevice_Check(device.ptr())) return t.device() == reinterpret_cast<THPDevice*>(device.ptr())->device;
    return py::cast(t.device()).equal(device);
}

bool is_readable(const at::Tensor& t, py::handle device) {
    return t.scalar_type() == at::kHalf && is_on(t, device) && t.layout() == at::kStrided && t.is_contiguous() &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

py::object address(const at::Tensor& t) { return py::reinterpret_steal<py::object>(PyLong_FromVoidPtr(t.data_ptr())); }

}  // namespace

bool all_bare(py::handle cls, const py::sequence& modules) {
    for (py::handle m : modules) {
        if (!is_bare(m.ptr(), cls.ptr())) return false;
    }
    return true;
}

bool children_bare(py::handle cls, const py::sequence& modules, const py::str& name) {
    for (py::handle m : modules) {
        if (!is_bare(attribute(m.ptr(), name.ptr()).ptr(), cls.ptr())) return false;
    }
    return true;
}

py::object rotary_tables(const py::sequence& layers, py::handle rotary, py::handle device) {
    py::list out;
    for (py::handle layer : layers) {
        const py::object r = attribute(layer.ptr(), names().rotary);
        if (!is_bare(r.ptr(), rotary.ptr())) return py::none();
        PyObject* own = own_dict(r.ptr());
        PyObject* buffers = get(own, names().buffers);
        if (get(own, names().table) || !buffers || !PyDict_CheckExact(buffers)) return py::none();
        PyObject* table = get(buffers, names().table);
        if (!table || !THPVariable_Check(table)) return py::none();
        const py::object width = attribute(r.ptr(), names().head_size);
        if (!py::bool_(attribute(r.ptr(), names().neox)) || !attribute(r.ptr(), names().rotary_dim).equal(width) ||
            !width.equal(attribute(layer.ptr(), names().head_dim))) {
            return py::none();
        }
        const at::Tensor& t = THPVariable_Unpack(table);
        if (t.dim() != 2 || t.size(1) != 128 || !is_readable(t, device)) return py::none();
        out.append(py::handle(table));
    }
    return std::move(out);
}

py::object linear_weights(const py::sequence& modules, py::handle linear, py::handle parameter, int64_t n_out, int64_t n_in,
                          py::handle device, bool grad) {
    py::list out, kept;
    for (py::handle m : modules) {
        if (!is_bare(m.ptr(), linear.ptr())) return py::none();
        PyObject* own = own_dict(m.ptr());
        if (get(own, names().weight) || get(own, names().bias)) return py::none();   // what hides the registered ones
        PyObject* parameters = get(own, names().parameters);
        if (!parameters || !PyDict_CheckExact(parameters)) return py::none();
        PyObject *w = get(parameters, names().weight), *b = get(parameters, names().bias);
        if (!w || reinterpret_cast<PyObject*>(Py_TYPE(w)) != parameter.ptr() || b != Py_None) return py::none();
        const at::Tensor& t = THPVariable_Unpack(w);
        if (t.dim() != 2 || t.size(1) != n_in || (n_out >= 0 && t.size(0) != n_out) || !is_readable(t, device) ||
            (grad && t.requires_grad())) {
            return py::none();
        }
        out.append(address(t));
        kept.append(py::handle(w));
    }
    return py::make_tuple(out, kept);
}

py::object parameter_addresses(const py::sequence& tensors, py::handle parameter, const std::vector<int64_t>& shape,
                               py::handle device) {
    py::list out;
    for (py::handle w : tensors) {
        if (reinterpret_cast<PyObject*>(Py_TYPE(w.ptr())) != parameter.ptr()) return py::none();
        const at::Tensor& t = THPVariable_Unpack(w.ptr());
        if (t.sizes() != at::IntArrayRef(shape) || !is_readable(t, device)) return py::none();
        out.append(address(t));
    }
    return std::move(out);
}

}  // namespace GPT

#pragma once

#include <pybind11/pybind11.h>
#include <torch/extension.h>

#include <vector>

namespace GPT {

namespace py = pybind11;

// Every module is a `cls` and nothing hangs on it that a call would also run (hooks, a patched forward).
bool all_bare(py::handle cls, const py::sequence& modules);

// The same of what the modules have under a name.
bool children_bare(py::handle cls, const py::sequence& modules, const py::str& name);

// The tables of the layers' rotary modules, if each is a bare `rotary` over whole heads in NeoX style, nothing hides its
// table, and the projection kernels read such a table (contiguous, 16-byte aligned fp16 [max_position, 128] on the
// device); None otherwise.
py::object rotary_tables(const py::sequence& layers, py::handle rotary, py::handle device);

// (addresses of the modules' weights, the weights), if what each computes of fp16 rows [..., n_in] on the device is exactly their
// product with a weight [n_out (-1: any), n_in] that the projection kernels read; None otherwise.
py::object linear_weights(const py::sequence& modules, py::handle linear, py::handle parameter, int64_t n_out, int64_t n_in,
                          py::handle device, bool grad);

// The tensors' addresses, if all are plain fp16 parameters of the shape, contiguous and 16-byte aligned on the device.
py::object parameter_addresses(const py::sequence& tensors, py::handle parameter, const std::vector<int64_t>& shape,
                               py::handle device);

}  // namespace GPT

// What the parts of the extension module share (native.cpp, native_mlp.cpp).
#pragma once

#include <algorithm>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>

#include "tk3d.h"

namespace tk3d {

using at::Tensor;
using torch::autograd::variable_list;

[[noreturn]] inline void fail(const std::string &message) { throw std::runtime_error(message); }

inline void done(int code, const char *what)
{
    if (code != TK3D_OK)
        fail(std::string(what) + " failed: " + tk3d_error_string(code) + " (code " +
             std::to_string(code) + ")");
}

inline void *stream_of(const Tensor &t)
{
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// Makes the tensor's GPU the current one (kernels, allocations and streams follow it).
using OnDeviceOf = c10::OptionalDeviceGuard;

// Whether the tensor is what its pointer and sizes say: no subclass that dispatches in Python, no
// wrapper of a function transform, no pending conjugation, and no forward-mode tangent.
bool plain(const Tensor &t);
// A function transform (torch.func), a dispatch mode or a tracer is active: it has to see the operators.
bool watched();
// Saved tensors come back through hooks, which may lay them out anew.
variable_list dense(variable_list saved);

variable_list mlp(Tensor x, Tensor x2, const Tensor &xyz, const Tensor &centre, const Tensor &index,
                  std::vector<Tensor> params, std::vector<Tensor> buffers, std::vector<double> eps,
                  std::vector<double> momentum, bool training, int64_t pool);

Tensor edge_lists(const Tensor &index, int64_t n);
Tensor edge_conv(const Tensor &x, const Tensor &index, const Tensor &lists,
                 const std::vector<Tensor> &params, const std::vector<Tensor> &buffers, double eps,
                 double momentum, bool training);

}  // namespace tk3d

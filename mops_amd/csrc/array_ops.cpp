// The functions of the mops_amd package on ROCm tensors, natively: what
// mops_amd/ops.py does for tensors that need no preparation, in 2 us beside the
// launch instead of 20 to 35 us of interpreter and ctypes.
//
// A function here looks at its arguments and either does the whole call or
// returns None, and then ops.py does it: anything but plain contiguous tensors
// of the expected dimensions and types on one device (numpy arrays, host
// tensors, 64-bit indices, a missing argument), and every call that fails, so
// that conversions and error messages are written down once, there.
#include <Python.h>

#include <array>

#include <torch/csrc/autograd/python_variable.h>

#include "mops.hpp"

#include "torch_tensors.hpp"

namespace {

using namespace mops::amd::torch_tensors;

/// One tensor argument: floating point or int32, and its dimensions.
struct Kind {
    bool index;
    int64_t dimensions;
};
constexpr Kind R1{false, 1}, R2{false, 2}, R3{false, 3}, I1{true, 1}, I2{true, 2};

/// The tensors among `arguments`, if all of them are what a kernel can take as it is.
template <size_t N> struct Inputs {
    std::array<const at::Tensor*, N> tensor;

    bool take(PyObject* const* arguments, const std::array<Kind, N>& kinds) {
        for (size_t i = 0; i < N; i++) {
            if (!THPVariable_CheckExact(arguments[i])) {
                return false;
            }
            const at::Tensor& t = THPVariable_Unpack(arguments[i]);
            if (!t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.is_neg() ||
                t.dim() != kinds[i].dimensions || !t.is_contiguous()) {
                return false;
            }
            if (i == 0 && t.scalar_type() != at::kFloat && t.scalar_type() != at::kDouble) {
                return false; // (the first tensor of every function is a floating-point one)
            }
            if (i > 0 && (t.device() != tensor[0]->device() ||
                          t.scalar_type() != (kinds[i].index ? at::kInt : tensor[0]->scalar_type()))) {
                return false;
            }
            tensor[i] = &t;
        }
        return true;
    }

    const at::Tensor& operator[](size_t i) const { return *tensor[i]; }
};

/// Which outputs are wanted: N flags, True or False.
template <size_t N> bool flags(PyObject* const* arguments, std::array<bool, N>& want) {
    for (size_t i = 0; i < N; i++) {
        if (!PyBool_Check(arguments[i])) {
            return false;
        }
        want[i] = arguments[i] == Py_True;
    }
    return true;
}
at::Tensor like_if(bool want, const at::Tensor& like) { return want ? new_like(like) : at::Tensor(); }

PyObject* wrap(const at::Tensor& tensor) {
    if (!tensor.defined()) {
        Py_RETURN_NONE;
    }
    return THPVariable_Wrap(tensor);
}
template <size_t N> PyObject* wrap(const std::array<at::Tensor, N>& tensors) {
    PyObject* tuple = PyTuple_New(N);
    for (size_t i = 0; tuple != nullptr && i < N; i++) {
        PyTuple_SET_ITEM(tuple, i, wrap(tensors[i]));
    }
    return tuple;
}

/// outputs(), then call(zero of the element type, outputs) on the tensors' stream and without the
/// interpreter lock; None when anything goes wrong.
template <typename Outputs, typename Call> PyObject* run(const at::Tensor& like, Outputs&& outputs, Call&& call) {
    try {
        OnTorchStream stream(like);
        auto results = outputs();
        PyThreadState* state = PyEval_SaveThread();
        try {
            by_dtype(like, [&](auto zero) { call(zero, results); });
        } catch (...) {
            PyEval_RestoreThread(state);
            Py_RETURN_NONE;
        }
        PyEval_RestoreThread(state);
        return wrap(results);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

/// An output size: a Python integer that fits.
bool size_of(PyObject* object, int64_t& size) {
    if (!PyLong_CheckExact(object)) {
        return false;
    }
    size = PyLong_AsLongLong(object);
    if (PyErr_Occurred() != nullptr) {
        PyErr_Clear();
        return false;
    }
    return size >= 0;
}

// ------------------------------------------------------------------- HPE ----
PyObject* hpe(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<3> t; // A C indices_A
    if (n != 3 || !t.take(arguments, {R2, R1, I2})) {
        Py_RETURN_NONE;
    }
    return run(t[0], [&] { return new_tensor({t[0].size(0)}, t[0]); }, [&](auto zero, at::Tensor& output) {
        using T = decltype(zero);
        mops::cuda::homogeneous_polynomial_evaluation<T>(
            view<T, 1>(output, "output"), view<T, 2>(t[0], "A"), view<T, 1>(t[1], "C"),
            view<int32_t, 2>(t[2], "indices_A")
        );
    });
}

PyObject* hpe_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<4> t; // grad_output A C indices_A
    std::array<bool, 1> want;
    if (n != 5 || !t.take(arguments, {R1, R2, R1, I2}) || !flags(arguments + 4, want)) {
        Py_RETURN_NONE;
    }
    return run(t[0], [&] { return like_if(want[0], t[1]); }, [&](auto zero, at::Tensor& grad_A) {
        using T = decltype(zero);
        mops::cuda::homogeneous_polynomial_evaluation_vjp<T>(
            view<T, 2>(grad_A, "grad_A"), view<T, 1>(t[0], "grad_output"), view<T, 2>(t[1], "A"),
            view<T, 1>(t[2], "C"), view<int32_t, 2>(t[3], "indices_A")
        );
    });
}

PyObject* hpe_vjp_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<5> t; // grad_grad_A grad_output A C indices_A
    std::array<bool, 2> want;
    if (n != 7 || !t.take(arguments, {R2, R1, R2, R1, I2}) || !flags(arguments + 5, want)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0], [&] { return std::array<at::Tensor, 2>{like_if(want[0], t[1]), like_if(want[1], t[2])}; },
        [&](auto zero, auto& out) {
            using T = decltype(zero);
            mops::cuda::homogeneous_polynomial_evaluation_vjp_vjp<T>(
                view<T, 1>(out[0], "grad_grad_output"), view<T, 2>(out[1], "grad_A_2"),
                view<T, 2>(t[0], "grad_grad_A"), view<T, 1>(t[1], "grad_output"), view<T, 2>(t[2], "A"),
                view<T, 1>(t[3], "C"), view<int32_t, 2>(t[4], "indices_A")
            );
        }
    );
}

// ------------------------------------------------------------------- SAP ----
PyObject* sap(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<6> t; // A B C indices_A indices_B indices_output
    int64_t size;
    if (n != 7 || !t.take(arguments, {R2, R2, R1, I1, I1, I1}) || !size_of(arguments[6], size)) {
        Py_RETURN_NONE;
    }
    return run(t[0], [&] { return new_tensor({t[0].size(0), size}, t[0]); }, [&](auto zero, at::Tensor& output) {
        using T = decltype(zero);
        mops::cuda::sparse_accumulation_of_products<T>(
            view<T, 2>(output, "output"), view<T, 2>(t[0], "A"), view<T, 2>(t[1], "B"), view<T, 1>(t[2], "C"),
            view<int32_t, 1>(t[3], "indices_A"), view<int32_t, 1>(t[4], "indices_B"),
            view<int32_t, 1>(t[5], "indices_output")
        );
    });
}

PyObject* sap_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<7> t; // grad_output A B C indices_A indices_B indices_output
    std::array<bool, 2> want;
    if (n != 9 || !t.take(arguments, {R2, R2, R2, R1, I1, I1, I1}) || !flags(arguments + 7, want)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0], [&] { return std::array<at::Tensor, 2>{like_if(want[0], t[1]), like_if(want[1], t[2])}; },
        [&](auto zero, auto& out) {
            using T = decltype(zero);
            mops::cuda::sparse_accumulation_of_products_vjp<T>(
                view<T, 2>(out[0], "grad_A"), view<T, 2>(out[1], "grad_B"), view<T, 2>(t[0], "grad_output"),
                view<T, 2>(t[1], "A"), view<T, 2>(t[2], "B"), view<T, 1>(t[3], "C"),
                view<int32_t, 1>(t[4], "indices_A"), view<int32_t, 1>(t[5], "indices_B"),
                view<int32_t, 1>(t[6], "indices_output")
            );
        }
    );
}

PyObject* sap_vjp_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<9> t; // grad_grad_A grad_grad_B grad_output A B C indices_A indices_B indices_output
    std::array<bool, 3> want;
    if (n != 12 || !t.take(arguments, {R2, R2, R2, R2, R2, R1, I1, I1, I1}) || !flags(arguments + 9, want)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0],
        [&] {
            return std::array<at::Tensor, 3>{like_if(want[0], t[2]), like_if(want[1], t[3]), like_if(want[2], t[4])};
        },
        [&](auto zero, auto& out) {
            using T = decltype(zero);
            mops::cuda::sparse_accumulation_of_products_vjp_vjp<T>(
                view<T, 2>(out[0], "grad_grad_output"), view<T, 2>(out[1], "grad_A_2"),
                view<T, 2>(out[2], "grad_B_2"), view<T, 2>(t[0], "grad_grad_A"), view<T, 2>(t[1], "grad_grad_B"),
                view<T, 2>(t[2], "grad_output"), view<T, 2>(t[3], "A"), view<T, 2>(t[4], "B"), view<T, 1>(t[5], "C"),
                view<int32_t, 1>(t[6], "indices_A"), view<int32_t, 1>(t[7], "indices_B"),
                view<int32_t, 1>(t[8], "indices_output")
            );
        }
    );
}

// ------------------------------------------------------------------ OPSA ----
PyObject* opsa(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<3> t; // A B indices_output
    int64_t size;
    if (n != 4 || !t.take(arguments, {R2, R2, I1}) || !size_of(arguments[3], size)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0], [&] { return new_tensor({size, t[0].size(1), t[1].size(1)}, t[0]); },
        [&](auto zero, at::Tensor& output) {
            using T = decltype(zero);
            mops::cuda::outer_product_scatter_add<T>(
                view<T, 3>(output, "output"), view<T, 2>(t[0], "A"), view<T, 2>(t[1], "B"),
                view<int32_t, 1>(t[2], "indices_output")
            );
        }
    );
}

PyObject* opsa_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<4> t; // grad_output A B indices_output
    std::array<bool, 2> want;
    if (n != 6 || !t.take(arguments, {R3, R2, R2, I1}) || !flags(arguments + 4, want)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0], [&] { return std::array<at::Tensor, 2>{like_if(want[0], t[1]), like_if(want[1], t[2])}; },
        [&](auto zero, auto& out) {
            using T = decltype(zero);
            mops::cuda::outer_product_scatter_add_vjp<T>(
                view<T, 2>(out[0], "grad_A"), view<T, 2>(out[1], "grad_B"), view<T, 3>(t[0], "grad_output"),
                view<T, 2>(t[1], "A"), view<T, 2>(t[2], "B"), view<int32_t, 1>(t[3], "indices_output")
            );
        }
    );
}

PyObject* opsa_vjp_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<6> t; // grad_grad_A grad_grad_B grad_output A B indices_output
    std::array<bool, 3> want;
    if (n != 9 || !t.take(arguments, {R2, R2, R3, R2, R2, I1}) || !flags(arguments + 6, want)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0],
        [&] {
            return std::array<at::Tensor, 3>{like_if(want[0], t[2]), like_if(want[1], t[3]), like_if(want[2], t[4])};
        },
        [&](auto zero, auto& out) {
            using T = decltype(zero);
            mops::cuda::outer_product_scatter_add_vjp_vjp<T>(
                view<T, 3>(out[0], "grad_grad_output"), view<T, 2>(out[1], "grad_A_2"),
                view<T, 2>(out[2], "grad_B_2"), view<T, 2>(t[0], "grad_grad_A"), view<T, 2>(t[1], "grad_grad_B"),
                view<T, 3>(t[2], "grad_output"), view<T, 2>(t[3], "A"), view<T, 2>(t[4], "B"),
                view<int32_t, 1>(t[5], "indices_output")
            );
        }
    );
}

// ----------------------------------------------------------------- OPSAW ----
PyObject* opsaw(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<5> t; // A B W indices_W indices_output
    if (n != 5 || !t.take(arguments, {R2, R2, R2, I1, I1})) {
        Py_RETURN_NONE;
    }
    return run(
        t[0], [&] { return new_tensor({t[2].size(0), t[0].size(1), t[1].size(1)}, t[0]); },
        [&](auto zero, at::Tensor& output) {
            using T = decltype(zero);
            mops::cuda::outer_product_scatter_add_with_weights<T>(
                view<T, 3>(output, "output"), view<T, 2>(t[0], "A"), view<T, 2>(t[1], "B"), view<T, 2>(t[2], "W"),
                view<int32_t, 1>(t[3], "indices_W"), view<int32_t, 1>(t[4], "indices_output")
            );
        }
    );
}

PyObject* opsaw_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<6> t; // grad_output A B W indices_W indices_output
    std::array<bool, 3> want;
    if (n != 9 || !t.take(arguments, {R3, R2, R2, R2, I1, I1}) || !flags(arguments + 6, want)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0],
        [&] {
            return std::array<at::Tensor, 3>{like_if(want[0], t[1]), like_if(want[1], t[2]), like_if(want[2], t[3])};
        },
        [&](auto zero, auto& out) {
            using T = decltype(zero);
            mops::cuda::outer_product_scatter_add_with_weights_vjp<T>(
                view<T, 2>(out[0], "grad_A"), view<T, 2>(out[1], "grad_B"), view<T, 2>(out[2], "grad_W"),
                view<T, 3>(t[0], "grad_output"), view<T, 2>(t[1], "A"), view<T, 2>(t[2], "B"), view<T, 2>(t[3], "W"),
                view<int32_t, 1>(t[4], "indices_W"), view<int32_t, 1>(t[5], "indices_output")
            );
        }
    );
}

// ----------------------------------------------------------------- SASAW ----
PyObject* sasaw(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<9> t; // A B C W indices_A indices_W_1 indices_W_2 indices_output_1 indices_output_2
    int64_t size;
    if (n != 10 || !t.take(arguments, {R2, R2, R1, R3, I1, I1, I1, I1, I1}) || !size_of(arguments[9], size)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0], [&] { return new_tensor({t[3].size(0), size, t[1].size(1)}, t[0]); },
        [&](auto zero, at::Tensor& output) {
            using T = decltype(zero);
            mops::cuda::sparse_accumulation_scatter_add_with_weights<T>(
                view<T, 3>(output, "output"), view<T, 2>(t[0], "A"), view<T, 2>(t[1], "B"), view<T, 1>(t[2], "C"),
                view<T, 3>(t[3], "W"), view<int32_t, 1>(t[4], "indices_A"), view<int32_t, 1>(t[5], "indices_W_1"),
                view<int32_t, 1>(t[6], "indices_W_2"), view<int32_t, 1>(t[7], "indices_output_1"),
                view<int32_t, 1>(t[8], "indices_output_2")
            );
        }
    );
}

PyObject* sasaw_vjp(PyObject*, PyObject* const* arguments, Py_ssize_t n) {
    Inputs<10> t; // grad_output A B C W indices_A indices_W_1 indices_W_2 indices_output_1 indices_output_2
    std::array<bool, 3> want;
    if (n != 13 || !t.take(arguments, {R3, R2, R2, R1, R3, I1, I1, I1, I1, I1}) || !flags(arguments + 10, want)) {
        Py_RETURN_NONE;
    }
    return run(
        t[0],
        [&] {
            return std::array<at::Tensor, 3>{like_if(want[0], t[1]), like_if(want[1], t[2]), like_if(want[2], t[4])};
        },
        [&](auto zero, auto& out) {
            using T = decltype(zero);
            mops::cuda::sparse_accumulation_scatter_add_with_weights_vjp<T>(
                view<T, 2>(out[0], "grad_A"), view<T, 2>(out[1], "grad_B"), view<T, 3>(out[2], "grad_W"),
                view<T, 3>(t[0], "grad_output"), view<T, 2>(t[1], "A"), view<T, 2>(t[2], "B"), view<T, 1>(t[3], "C"),
                view<T, 3>(t[4], "W"), view<int32_t, 1>(t[5], "indices_A"), view<int32_t, 1>(t[6], "indices_W_1"),
                view<int32_t, 1>(t[7], "indices_W_2"), view<int32_t, 1>(t[8], "indices_output_1"),
                view<int32_t, 1>(t[9], "indices_output_2")
            );
        }
    );
}

#define MOPS_METHOD(NAME, FUNCTION)                                                                 \
    {NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(FUNCTION)), METH_FASTCALL, nullptr}
PyMethodDef METHODS[] = {
    MOPS_METHOD("homogeneous_polynomial_evaluation", hpe),
    MOPS_METHOD("homogeneous_polynomial_evaluation_vjp", hpe_vjp),
    MOPS_METHOD("homogeneous_polynomial_evaluation_vjp_vjp", hpe_vjp_vjp),
    MOPS_METHOD("sparse_accumulation_of_products", sap),
    MOPS_METHOD("sparse_accumulation_of_products_vjp", sap_vjp),
    MOPS_METHOD("sparse_accumulation_of_products_vjp_vjp", sap_vjp_vjp),
    MOPS_METHOD("outer_product_scatter_add", opsa),
    MOPS_METHOD("outer_product_scatter_add_vjp", opsa_vjp),
    MOPS_METHOD("outer_product_scatter_add_vjp_vjp", opsa_vjp_vjp),
    MOPS_METHOD("outer_product_scatter_add_with_weights", opsaw),
    MOPS_METHOD("outer_product_scatter_add_with_weights_vjp", opsaw_vjp),
    MOPS_METHOD("sparse_accumulation_scatter_add_with_weights", sasaw),
    MOPS_METHOD("sparse_accumulation_scatter_add_with_weights_vjp", sasaw_vjp),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "_array_ops", nullptr, -1, METHODS, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__array_ops() { return PyModule_Create(&MODULE); }

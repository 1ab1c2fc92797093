// The quantizers' calls on plain GPU tensors without the Python between a call and its launch.
//
// A quantizer call on 2000 rows is a 3.9 us kernel behind 3.3 us of the runtime's launch; checking the tensors, reading their
// addresses and marshalling the arguments in Python took 3.0 us more.  Each function here answers 1 when it has queued the work,
// a negative status of the library, or 0 when something about the tensors is not plain (another device, dtype, layout or
// size, a subclass): the Python wrapper then takes the call from the beginning, with its staging and its error messages.
#include <Python.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "sgnn.h"

namespace {

decltype(&sgnn_quant_pack_rows_f32) quant_f32;
decltype(&sgnn_quant_pack_rows_wire_f32) quant_wire;
decltype(&sgnn_unpack_dequant_rows_f32) dequant_f32;
decltype(&sgnn_unpack_dequant_rows_wire_f32) dequant_wire;

// Other Python threads run while this lives.  (Taken back on every way out: the library reports errors through strings, which
// may throw.)
struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

const at::Tensor *plain(PyObject *o, int device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.is_cuda() && t.has_storage() && t.get_device() == device && t.is_contiguous() ? &t : nullptr;
}

// (fp32 rows, packed rows, parameters, the segments' rows and packed rows (tensors of P + 1), rows, packed rows, bits); QUANT: from
// the rows to the packed rows, else back.
template <bool QUANT>
PyObject *rows(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    if (n_args != 8) return PyLong_FromLong(0);
    const int64_t n_rows = PyLong_AsLongLong(args[5]), n_packed = PyLong_AsLongLong(args[6]);
    const long bits = PyLong_AsLong(args[7]);
    if (PyErr_Occurred()) { PyErr_Clear(); return PyLong_FromLong(0); }
    try {
        const int device = c10::hip::current_device();
        const at::Tensor *x = plain(args[0], device), *q = plain(args[1], device), *p = plain(args[2], device),
                         *seg = plain(args[3], device), *pseg = plain(args[4], device);
        if (!x || !q || !p || !seg || !pseg || x->scalar_type() != at::kFloat || q->scalar_type() != at::kByte || x->dim() != 2 ||
            seg->scalar_type() != at::kInt || pseg->scalar_type() != at::kInt || seg->numel() < 1 || pseg->numel() != seg->numel())
            return PyLong_FromLong(0);
        const int P = (int)seg->numel() - 1;
        const int32_t *sp = seg->const_data_ptr<int32_t>(), *psp = pseg->const_data_ptr<int32_t>();
        const bool bf16 = p->scalar_type() == at::kBFloat16;
        const int64_t F = x->size(1);
        if ((!bf16 && p->scalar_type() != at::kFloat) || x->size(0) != n_rows || q->numel() < n_packed * F || p->numel() < n_rows * 2)
            return PyLong_FromLong(0);
        const hipStream_t st = c10::hip::getCurrentHIPStream(device).stream();
        int rc;
        if constexpr (QUANT) {
            const float *xp = x->const_data_ptr<float>();
            uint8_t *qp = q->mutable_data_ptr<uint8_t>();
            void *pp = p->mutable_data_ptr();
            const WithoutGil unlocked;
            rc = bf16 ? quant_wire(xp, F, nullptr, n_rows, qp, pp, 1, sp, psp, P, n_rows, n_packed, F, (int)bits, st)
                      : quant_f32(xp, qp, static_cast<float *>(pp), sp, psp, P, n_rows, n_packed, F, (int)bits, st);
        } else {
            const uint8_t *qp = q->const_data_ptr<uint8_t>();
            float *xp = x->mutable_data_ptr<float>();
            const void *pp = p->const_data_ptr();
            const WithoutGil unlocked;
            rc = bf16 ? dequant_wire(qp, xp, pp, 1, sp, psp, P, n_rows, n_packed, F, (int)bits, st)
                      : dequant_f32(qp, xp, static_cast<const float *>(pp), sp, psp, P, n_rows, n_packed, F, (int)bits, st);
        }
        return PyLong_FromLong(rc < 0 ? rc : 1);
    } catch (...) {
        return PyLong_FromLong(0);
    }
}

// The library's entry points, by address: the library is already loaded, from the package's own path.
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    if (n_args != 4) {
        PyErr_SetString(PyExc_TypeError, "bind takes four addresses");
        return nullptr;
    }
    void *p[4];
    for (int i = 0; i < 4; ++i) p[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
    quant_f32 = reinterpret_cast<decltype(quant_f32)>(p[0]);
    quant_wire = reinterpret_cast<decltype(quant_wire)>(p[1]);
    dequant_f32 = reinterpret_cast<decltype(dequant_f32)>(p[2]);
    dequant_wire = reinterpret_cast<decltype(dequant_wire)>(p[3]);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(bind)), METH_FASTCALL, nullptr},
    {"quant_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(rows<true>)), METH_FASTCALL, nullptr},
    {"dequant_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(rows<false>)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_direct", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__direct() { return PyModule_Create(&module); }

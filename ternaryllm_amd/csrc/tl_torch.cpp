// The short way from a torch call to a product: what ops.spmm and ops.mlp_gate_up do in Python, for the plain calls (ordinary
// tensors on the weight's device, one of the library's types, rows or one K-major matrix, no workspace or one that is there).
// A call that is anything else gets None, and Python's general path, which also words the errors.
//
// Bound by the host: one fp16 row 4096 x 4096 is 4 us of kernel; through Python's checks, ctypes and stream objects the call took
// 18.6 us, this way 7.1 (another launch before it has ended; 2.5 us of it are the launch).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "ternary_spmm.h"

namespace {

// The library's entry points, as Python loaded it (init).
decltype(&tl_spmm) g_spmm;
decltype(&tl_spmm_workspace) g_workspace;
decltype(&tl_mlp_gate_up) g_gate_up;
decltype(&tl_mlp_gate_up_few) g_gate_up_few;
PyObject* g_workspaces;  // {(device index, stream): uint8 tensor}: the scratch of ops

int type_code(const at::Tensor& t)
{
    return t.scalar_type() == at::kHalf ? TL_F16 : t.scalar_type() == at::kFloat ? TL_F32 : -1;
}

// A tensor with no class, mode or wrapper of its own between the caller and its memory; null for None and for anything else.
const at::Tensor* plain(PyObject* o)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.layout() == at::kStrided && t.is_cuda() && !t.is_neg() && !t.is_conj() && t.has_storage() ? &t : nullptr;
}

struct Rows {
    int64_t M = 0, ld = 0;
    int layout = TL_X_ROW_MAJOR;
};

// x as the library's activations of K rows of a weight: [.., K] in uniform rows, or, kmajor, [K, M] or [1, K, M].
bool geometry(const at::Tensor& x, int64_t K, bool kmajor, Rows* r)
{
    const int64_t dims = x.dim();
    if (dims < 1 || dims > 3) return false;
    if (kmajor) {
        if (dims < 2 || (dims == 3 && x.size(0) != 1) || x.size(-2) != K || x.stride(-1) != 1) return false;
        r->M = x.size(-1);
        r->ld = K > 1 ? x.stride(-2) : std::max<int64_t>(r->M, 1);
        r->layout = TL_X_K_MAJOR;
        return r->M > 0;
    }
    if (x.size(-1) != K || (dims != 2 && !x.is_contiguous()) || x.stride(-1) != 1) return false;
    r->M = dims == 1 ? 1 : dims == 2 ? x.size(0) : x.size(0) * x.size(1);
    r->ld = dims == 2 && r->M > 1 ? x.stride(0) : std::max<int64_t>(K, 1);
    return r->M > 0;
}

bool scale_fits(PyObject* o, const at::Tensor** scale, int64_t N, c10::Device device)
{
    *scale = nullptr;
    if (o == Py_None) return true;
    const at::Tensor* s = plain(o);
    if (!s || s->device() != device || s->numel() != N || !s->is_contiguous() || type_code(*s) < 0) return false;
    *scale = s;
    return true;
}

// The call's workspace (kept until the call has been made, whatever another thread does to the dict): false where Python has
// to make one first.
bool workspace(const tl_layout_header* header, const Rows& r, int x_type, c10::Device device, void* stream, at::Tensor* ws)
{
    int64_t need = 0;
    if (g_workspace(header, r.M, x_type, r.layout, &need) != TL_OK) return false;
    if (need == 0) return true;
    PyObject* key = Py_BuildValue("(iK)", (int)device.index(), (unsigned long long)(uintptr_t)stream);
    if (!key) throw python_error();
    PyObject* found = PyDict_GetItemWithError(g_workspaces, key);  // borrowed
    Py_DECREF(key);
    if (!found && PyErr_Occurred()) throw python_error();
    if (!found || !THPVariable_Check(found)) return false;
    const at::Tensor& t = THPVariable_Unpack(found);
    if (t.numel() < need) return false;
    *ws = t;
    return true;
}

void* current_stream(c10::Device device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

at::Tensor output(const at::Tensor& x, const Rows& r, int64_t N, bool kmajor)
{
    c10::SmallVector<int64_t, 3> shape(x.sizes().begin(), x.sizes().end());
    if (kmajor) shape[shape.size() - 2] = r.M;
    shape.back() = N;
    return at::empty(shape, x.options().requires_grad(false));
}

const tl_layout_header* header_at(PyObject* address) { return static_cast<const tl_layout_header*>(PyLong_AsVoidPtr(address)); }

// product(header address, blob, x, scale or None, kmajor or None: x of K values a row is rows) -> tensor or None
PyObject* product(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    if (count != 5) {
        PyErr_SetString(PyExc_TypeError, "product takes five arguments");
        return nullptr;
    }
    const tl_layout_header* header = header_at(args[0]);
    const at::Tensor *blob = plain(args[1]), *x = plain(args[2]), *scale;
    const bool kmajor = args[4] == Py_None ? header && x && x->dim() > 0 && x->size(-1) != header->inners : args[4] == Py_True;
    Rows r;
    if (!header || !blob || !x || x->device() != blob->device() || type_code(*x) < 0 || !geometry(*x, header->inners, kmajor, &r) ||
        !scale_fits(args[3], &scale, header->columns, x->device()))
        Py_RETURN_NONE;
    const c10::DeviceGuard guard(x->device());
    void* stream = current_stream(x->device());
    at::Tensor ws;
    const int type = type_code(*x);
    if (!workspace(header, r, type, x->device(), stream, &ws)) Py_RETURN_NONE;
    at::Tensor y = output(*x, r, header->columns, kmajor);
    int rc;
    {
        const pybind11::gil_scoped_release no_gil;
        rc = g_spmm(header, blob->data_ptr(), x->data_ptr(), type, r.layout, r.ld, r.M, y.data_ptr(), type, header->columns,
                    scale ? scale->data_ptr() : nullptr, scale ? type_code(*scale) : TL_F32, ws.defined() ? ws.data_ptr() : nullptr,
                    ws.defined() ? ws.numel() : 0, stream);
    }
    if (rc != TL_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// gate_up(gate header, gate blob, up header, up blob, x, gate scale, up scale) -> silu(gate) * up, or None
PyObject* gate_up(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    if (count != 7) {
        PyErr_SetString(PyExc_TypeError, "gate_up takes seven arguments");
        return nullptr;
    }
    const tl_layout_header *g = header_at(args[0]), *u = header_at(args[2]);
    const at::Tensor *gb = plain(args[1]), *ub = plain(args[3]), *x = plain(args[4]), *gs, *us;
    Rows r;
    if (!g || !u || !gb || !ub || !x || x->device() != gb->device() || x->device() != ub->device() || type_code(*x) < 0 ||
        g->inners != u->inners || g->columns != u->columns || g->tile_rows != u->tile_rows || !geometry(*x, g->inners, false, &r) ||
        !scale_fits(args[5], &gs, g->columns, x->device()) || !scale_fits(args[6], &us, g->columns, x->device()) ||
        (gs == nullptr) != (us == nullptr) || (gs && type_code(*gs) != type_code(*us)))
        Py_RETURN_NONE;
    const bool few = r.M <= 48;
    if (few && (r.M < 2 || !g->off_codes || !u->off_codes)) Py_RETURN_NONE;
    const c10::DeviceGuard guard(x->device());
    void* stream = current_stream(x->device());
    at::Tensor ws;
    const int type = type_code(*x), scale_type = gs ? type_code(*gs) : TL_F32;
    if (!few && !workspace(g, r, type, x->device(), stream, &ws)) Py_RETURN_NONE;
    at::Tensor h = output(*x, r, g->columns, false);
    int rc;
    {
        const pybind11::gil_scoped_release no_gil;
        const void *gsp = gs ? gs->data_ptr() : nullptr, *usp = us ? us->data_ptr() : nullptr;
        rc = few ? g_gate_up_few(g, gb->data_ptr(), u, ub->data_ptr(), x->data_ptr(), type, TL_X_ROW_MAJOR, r.ld, r.M, h.data_ptr(), type, g->columns,
                                 gsp, usp, scale_type, TL_ACT_SILU_GATE, stream)
                 : g_gate_up(g, gb->data_ptr(), u, ub->data_ptr(), x->data_ptr(), type, TL_X_ROW_MAJOR, r.ld, r.M, h.data_ptr(), type, g->columns,
                             gsp, usp, scale_type, TL_ACT_SILU_GATE, ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? ws.numel() : 0, stream);
    }
    if (rc != TL_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(h));
    END_HANDLE_TH_ERRORS
}

// init(addresses of tl_spmm, tl_spmm_workspace, tl_mlp_gate_up, tl_mlp_gate_up_few, the scratch dict)
PyObject* init(PyObject*, PyObject* args)
{
    PyObject *spmm, *space, *both, *few, *dict;
    if (!PyArg_ParseTuple(args, "OOOOO!", &spmm, &space, &both, &few, &PyDict_Type, &dict)) return nullptr;
    g_spmm = reinterpret_cast<decltype(g_spmm)>(PyLong_AsVoidPtr(spmm));
    g_workspace = reinterpret_cast<decltype(g_workspace)>(PyLong_AsVoidPtr(space));
    g_gate_up = reinterpret_cast<decltype(g_gate_up)>(PyLong_AsVoidPtr(both));
    g_gate_up_few = reinterpret_cast<decltype(g_gate_up_few)>(PyLong_AsVoidPtr(few));
    if (PyErr_Occurred()) return nullptr;
    Py_INCREF(dict);
    g_workspaces = dict;
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"init", init, METH_VARARGS, "addresses of the library's entry points, and the scratch buffers"},
    {"product", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(product)), METH_FASTCALL, "x @ W * scale, or None"},
    {"gate_up", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gate_up)), METH_FASTCALL, "silu(x @ Wg) * (x @ Wu), or None"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_tl_torch", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tl_torch(void) { return PyModule_Create(&g_module); }

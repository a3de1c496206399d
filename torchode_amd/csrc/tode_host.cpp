// torchode_amd._host: what AutoDiffAdjoint.solve does around the kernel of a whole solve with a built-in term -- the argument
// block from the problem's tensors, the outputs from PyTorch's allocator, the launch, the views of the statistics while
// the kernel runs, and the wait -- as one call of a Python extension.  A small solve's kernel takes 25 to 75 microseconds, and
// the same steps in Python, one ctypes or tensor call each, took 23 ahead of the launch where they now take 9 (decay, float64,
// B = 256: 52 -> 40 us a solve; Lorenz to its end point, B = 40 009: 80 -> 67; perceptron, B = 4096: 109 -> 91).  No solver logic and
// no kernel: everything here ends in the C ABI of include/torchode_amd.h, and nothing is kept from one call for the next.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/torchode_amd.h"

namespace {

using at::Tensor;

struct PythonError {};  // (set already)

const Tensor &tensor(PyObject *o, const char *name) {
    if (THPVariable_Check(o)) return THPVariable_Unpack(o);
    PyErr_Format(PyExc_TypeError, "%s must be a tensor, got %s", name, Py_TYPE(o)->tp_name);
    throw PythonError();
}
double number(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PythonError();
    return v;
}
long long integer(PyObject *o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw PythonError();
    return v;
}
int dtype_code(at::ScalarType t) {
    TORCH_CHECK_NOT_IMPLEMENTED(t == at::kFloat || t == at::kDouble, "the kernels are built for float32 and float64 (got ", t, ")");
    return t == at::kFloat ? TODE_F32 : TODE_F64;
}
[[noreturn]] void library_error(const char *call, int rc) {
    PyErr_Format(PyExc_RuntimeError, "%s failed with code %d: %s", call, rc, tode_last_error());
    throw PythonError();
}

// The library waits for the GPU in it: other Python threads run meanwhile.
struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

PyObject *append(PyObject *tuple, Py_ssize_t i, PyObject *item) {
    if (!item) {
        Py_DECREF(tuple);
        throw PythonError();
    }
    PyTuple_SET_ITEM(tuple, i, item);
    return tuple;
}

// solve(y0, t_start, t_end, t_eval, dt0, params, shared_params, method, term, term_scalars, max_steps, allow_one_kernel, has_general, kind, dt_min,
//       dt_max, atol, rtol, pcoeff, icoeff, dcoeff, safety, factor_min, factor_max)
// -> (ys, n_steps, n_accepted, n_initialized, status, iterations), or None where no whole-solve kernel takes the problem
constexpr Py_ssize_t N_ARGS = 24;

PyObject *solve_(PyObject *const *arg) {
    const Tensor &y0_ = tensor(arg[0], "y0");
    const bool has_eval = arg[3] != Py_None, has_dt0 = arg[4] != Py_None, has_params = arg[5] != Py_None, has_shared = arg[6] != Py_None;
    const Tensor y0 = y0_.contiguous();
    // t_start / t_end are usually columns of t_eval: handed over with their stride
    auto column = [](const Tensor &t) { return t.stride(0) >= 1 ? t : t.contiguous(); };
    const Tensor t_start = column(tensor(arg[1], "t_start")), t_end = column(tensor(arg[2], "t_end"));
    const Tensor t_eval = has_eval ? tensor(arg[3], "t_eval").contiguous() : Tensor();
    const auto dtype = y0.scalar_type(), time_dtype = t_start.scalar_type();
    const Tensor dt0 = has_dt0 ? tensor(arg[4], "dt0").to(time_dtype).contiguous() : Tensor();
    const int64_t B = y0.size(0), F = y0.size(1), E = has_eval ? t_eval.size(1) : 0;
    Tensor params;
    if (has_params) {
        params = tensor(arg[5], "the term's parameters");
        if (params.device() != y0.device() || params.scalar_type() != dtype) params = params.to(y0.options());
        if (params.numel() == 0 && params.size(0) != B) params = params.new_empty({B, 0});  // a term without per-sample parameters
        if (params.dim() != 2 || params.size(0) != B) {
            PyErr_SetString(PyExc_AssertionError, "built-in term parameters do not match the batch size");
            throw PythonError();
        }
        params = params.contiguous();
    }
    const Tensor shared = has_shared ? tensor(arg[6], "the shared parameters") : Tensor();

    tode_solve_args a = {};
    const int data_code = dtype_code(dtype), time_code = dtype_code(time_dtype);
    a.dtype = data_code == time_code ? data_code : TODE_DTYPES(data_code, time_code);
    a.method = (int32_t)integer(arg[7]), a.term = (int32_t)integer(arg[8]);
    a.n_features = (int32_t)F, a.n_eval = (int32_t)E, a.n_params = has_params ? (int32_t)params.size(1) : 0;
    a.batch = B, a.max_steps = arg[10] == Py_None ? -1 : integer(arg[10]), a.iteration_cap = -1;
    const Py_ssize_t n_scalars = PyTuple_Check(arg[9]) ? PyTuple_GET_SIZE(arg[9]) : 0;
    for (Py_ssize_t i = 0; i < n_scalars && i < 4; ++i) a.term_scalars[i] = number(PyTuple_GET_ITEM(arg[9], i));
    a.y0 = y0.data_ptr();
    a.t_start = t_start.data_ptr(), a.t_end = t_end.data_ptr();
    a.t_start_stride = t_start.stride(0), a.t_end_stride = t_end.stride(0);
    a.t_eval = has_eval ? t_eval.data_ptr() : nullptr, a.dt0 = has_dt0 ? dt0.data_ptr() : nullptr;
    a.params = has_params && params.numel() > 0 ? params.data_ptr() : nullptr;
    a.shared_params = has_shared ? shared.data_ptr() : nullptr, a.n_shared_params = has_shared ? shared.numel() : 0;
    const int allow_one_kernel = PyObject_IsTrue(arg[11]), has_general = PyObject_IsTrue(arg[12]);
    if (allow_one_kernel < 0 || has_general < 0) throw PythonError();

    tode_controller c = {};
    c.kind = (int32_t)integer(arg[13]);
    c.has_dt_min = arg[14] != Py_None, c.has_dt_max = arg[15] != Py_None;
    c.dt_min = c.has_dt_min ? number(arg[14]) : 0.0, c.dt_max = c.has_dt_max ? number(arg[15]) : 0.0;
    double *const values[] = {&c.atol, &c.rtol, &c.pcoeff, &c.icoeff, &c.dcoeff, &c.safety, &c.factor_min, &c.factor_max};
    for (int i = 0; i < 8; ++i) *values[i] = number(arg[16 + i]);

    const c10::DeviceGuard guard(y0.device());
    void *const stream = (void *)c10::hip::getCurrentHIPStream(y0.device().index()).stream();
    const Tensor ys = at::empty({B, E > 0 ? E : 1, F}, y0.options());
    const Tensor out = at::empty({4, B}, y0.options().dtype(at::kLong));
    const Tensor y_idle = E == 0 ? at::empty({B, F}, y0.options()) : Tensor();
    a.ys = ys.data_ptr(), a.y_idle = E == 0 ? y_idle.data_ptr() : nullptr;
    int64_t *const stats = out.data_ptr<int64_t>();

    tode_solve_ticket ticket;
    int rc;
    {
        WithoutGil released;
        rc = tode_solve_builtin_begin(&a, &c, stats, stats + B, stats + 2 * B, stats + 3 * B, allow_one_kernel, stream, &ticket);
    }
    if (rc == TODE_E_UNSUPPORTED) Py_RETURN_NONE;  // no whole-solve kernel for this case: the caller takes the per-step or the operator path
    if (rc) library_error("tode_solve_builtin_begin", rc);
    struct End {  // (a ticket that was begun is ended, whatever happens in between)
        tode_solve_ticket &ticket;
        const tode_solve_args &a;
        const int64_t *stats;
        void *stream;
        int32_t flags[TODE_FLAG_WORDS];
        bool ended = false;
        int wait() {
            ended = true;
            WithoutGil released;
            return tode_solve_builtin_end(&ticket, &a, stats, stream, flags);
        }
        ~End() {
            if (!ended) (void)wait();
        }
    } end{ticket, a, stats, stream, {}};

    // while the kernel runs
    PyObject *result = PyTuple_New(6);
    if (!result) throw PythonError();
    append(result, 0, THPVariable_Wrap(ys));
    for (int64_t i = 0; i < 4; ++i) append(result, 1 + i, THPVariable_Wrap(out.select(0, i)));

    rc = end.wait();  // (the solve's one host synchronisation)
    const char *call = "tode_solve_builtin_end";
    int64_t iterations = end.flags[TODE_FLAG_MAX_ITERATIONS];
    if (rc == TODE_OK && end.flags[TODE_FLAG_NEEDS_GENERAL]) {
        if (!has_general) {
            Py_DECREF(result);
            Py_RETURN_NONE;
        }
        call = "tode_solve_builtin_auto";
        const int64_t bytes = tode_solve_workspace_bytes(&a);
        const Tensor workspace = at::empty({bytes}, y0.options().dtype(at::kByte));
        WithoutGil released;
        rc = tode_solve_builtin_auto(&a, &c, stats, stats + B, stats + 2 * B, stats + 3 * B, workspace.data_ptr(), bytes, 0, stream, &iterations);
    }
    if (rc) {
        Py_DECREF(result);
        library_error(call, rc);
    }
    return append(result, 5, PyLong_FromLongLong(iterations));
}

// stage(state, controller, i, y, t, k, stream): stage i of an iteration around a user's right-hand side (tode_step_stage): a node time
// and a stage input made like t and y, the launch that fills them, and (time, input) as the right-hand side's arguments.  k: the
// derivative of the stage before, contiguous and of y's shape and type, or None.  state, controller, stream: addresses.
PyObject *stage_(PyObject *const *arg) {
    tode_step_state *const s = (tode_step_state *)PyLong_AsVoidPtr(arg[0]);
    const tode_controller *const c = (const tode_controller *)PyLong_AsVoidPtr(arg[1]);
    const long long i = integer(arg[2]);
    void *const stream = arg[6] == Py_None ? nullptr : PyLong_AsVoidPtr(arg[6]);
    if (PyErr_Occurred()) throw PythonError();
    if (!s || !c || i < 1 || i > 6) {
        PyErr_SetString(PyExc_ValueError, "stage: null address or stage out of range");
        throw PythonError();
    }
    const Tensor &y = tensor(arg[3], "y"), &t = tensor(arg[4], "t");
    if (arg[5] != Py_None) {
        const Tensor &k = tensor(arg[5], "k");
        TORCH_CHECK_VALUE(k.scalar_type() == y.scalar_type() && k.device() == y.device() && k.sizes() == y.sizes() && k.is_contiguous(), "stage: k must be contiguous and of y's shape, type and device");
        s->k[i - 1] = k.data_ptr();
    }
    const Tensor input = at::empty(y.sizes(), y.options()), node = at::empty(t.sizes(), t.options());
    s->ystage[i] = input.data_ptr(), s->tnode = node.data_ptr();
    int rc;
    {
        WithoutGil released;
        rc = tode_step_stage(s, c, (int32_t)i, stream);
    }
    if (rc) library_error("tode_step_stage", rc);
    PyObject *result = PyTuple_New(2);
    if (!result) throw PythonError();
    append(result, 0, THPVariable_Wrap(node));
    return append(result, 1, THPVariable_Wrap(input));
}

template <Py_ssize_t N, PyObject *(*F)(PyObject *const *)> PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "takes %zd arguments, got %zd", N, n);
        return nullptr;
    }
    HANDLE_TH_ERRORS
    try {
        return F(args);
    } catch (const PythonError &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"solve", (PyCFunction)(void (*)())entry<N_ARGS, solve_>, METH_FASTCALL, "One whole solve with a built-in term (see torchode_amd.adjoints)."},
    {"stage", (PyCFunction)(void (*)())entry<7, stage_>, METH_FASTCALL, "One stage around a user's right-hand side (see torchode_amd.adjoints)."},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }

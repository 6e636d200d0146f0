// smat_amd.spmm as a function of an extension module: the same call as host.py makes through ctypes, for arguments of the types that programs pass.
//
// A small product is over sooner than the call that launches it.  Through ctypes a call was asked for by bytecode, address by address, and turned into C arguments by ctypes'
// table.  That -> here, us of the host a call, the runtime's launch among them, twenty in a row (band of 4096 rows and 64, N = 128): with a plan 5.1 to 5.4 -> 4.5, drop-in 5.3 to 5.5 -> 4.8.
// Anything else than plain arguments (numbers that are no int, a plan of another class, a wrong number of arguments) goes to the function in Python, which takes
// or refuses it as before.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

#include "../../../include/smat.h"

namespace {

decltype(&smat_spmm_bcsr_f16_ex) g_launch = nullptr;
decltype(&smat_spmm_bcsr_f16) g_launch_drop_in = nullptr;
PyObject *g_in_python = nullptr, *g_check = nullptr, *g_plan_type = nullptr;
PyObject *g_data_ptr = nullptr, *g_address = nullptr;

enum { VALS, ROW_PTR, COL_IDX, B, C_OUT, M, N, K, NNZB, PLAN, C_F32, KERNEL, STREAM, DROP_IN, B_ROW_MAJOR, N_ARGS };
const char *const NAMES[N_ARGS] = {"vals", "row_ptr", "col_idx", "B", "C_out", "M", "N", "K", "nnzb", "plan", "c_f32", "kernel", "stream", "drop_in", "b_row_major"};
PyObject *g_names[N_ARGS];

// 1: *out is the address; 0: not for here; -1: data_ptr() raised
int address_of(PyObject *o, void **out)
{
    if (o == Py_None) {
        *out = nullptr;
        return 1;
    }
    PyObject *const r = PyObject_VectorcallMethod(g_data_ptr, &o, 1 | PY_VECTORCALL_ARGUMENTS_OFFSET, nullptr);
    if (!r) return -1;
    const bool plain = PyLong_CheckExact(r);
    if (plain) *out = reinterpret_cast<void *>(PyLong_AsUnsignedLongLongMask(r));
    Py_DECREF(r);
    return plain;
}
bool flag_of(PyObject *o, bool *out)
{
    *out = o == Py_True;
    return o == Py_True || o == Py_False;
}

PyObject *spmm(PyObject *, PyObject *const *args, Py_ssize_t n, PyObject *kwnames)
{
    auto in_python = [&] { return PyObject_Vectorcall(g_in_python, args, (size_t)n, kwnames); };
    PyObject *a[N_ARGS] = {};
    if (n > N_ARGS) return in_python();
    for (Py_ssize_t i = 0; i < n; i++) a[i] = args[i];
    const Py_ssize_t named = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t i = 0; i < named; i++) {
        PyObject *const name = PyTuple_GET_ITEM(kwnames, i);
        int at = 0;
        while (at < N_ARGS && g_names[at] != name) at++; // names in source code are interned, as these are
        if (at == N_ARGS || a[at]) return in_python();
        a[at] = args[n + i];
    }
    for (int i = VALS; i <= NNZB; i++)
        if (!a[i]) return in_python();
    size_t size[4];
    for (int i = 0; i < 4; i++) {
        if (!PyLong_CheckExact(a[M + i])) return in_python();
        size[i] = (size_t)PyLong_AsUnsignedLongLongMask(a[M + i]);
    }
    bool c_f32 = false, drop_in = false, b_row_major = false;
    if ((a[C_F32] && !flag_of(a[C_F32], &c_f32)) || (a[DROP_IN] && !flag_of(a[DROP_IN], &drop_in)) || (a[B_ROW_MAJOR] && !flag_of(a[B_ROW_MAJOR], &b_row_major)))
        return in_python();
    long kernel = 0;
    void *stream = nullptr;
    if (a[KERNEL]) {
        if (!PyLong_CheckExact(a[KERNEL])) return in_python();
        int overflow;
        kernel = PyLong_AsLongAndOverflow(a[KERNEL], &overflow);
        if (overflow || kernel != (int32_t)kernel) return in_python();
    }
    if (a[STREAM] && a[STREAM] != Py_None) {
        if (!PyLong_CheckExact(a[STREAM])) return in_python();
        stream = reinterpret_cast<void *>(PyLong_AsUnsignedLongLongMask(a[STREAM]));
    }
    const smat_plan *plan = nullptr;
    if (a[PLAN] && a[PLAN] != Py_None) {
        if ((PyObject *)Py_TYPE(a[PLAN]) != g_plan_type) return in_python();
        PyObject *const h = PyObject_GetAttr(a[PLAN], g_address);
        if (!h) return nullptr;
        const bool plain = PyLong_CheckExact(h);
        if (plain) plan = static_cast<const smat_plan *>(reinterpret_cast<void *>(PyLong_AsUnsignedLongLongMask(h)));
        Py_DECREF(h);
        if (!plain) return in_python();
    }
    void *p[5];
    for (int i = 0; i < 5; i++) {
        const int r = address_of(a[VALS + i], &p[i]);
        if (r < 0) return nullptr;
        if (r == 0) return in_python();
    }
    int rc;
    Py_BEGIN_ALLOW_THREADS
    const auto *vals = static_cast<const uint16_t *>(p[0]), *b = static_cast<const uint16_t *>(p[3]);
    const auto *row_ptr = static_cast<const int32_t *>(p[1]), *col_idx = static_cast<const int32_t *>(p[2]);
    if (drop_in) {
        rc = g_launch_drop_in(vals, row_ptr, col_idx, b, static_cast<uint16_t *>(p[4]), size[0], size[1], size[2], size[3], nullptr, nullptr);
    } else {
        const smat_spmm_opts o = {b_row_major ? SMAT_B_ROW_MAJOR : SMAT_B_COL_MAJOR, c_f32 ? SMAT_C_F32 : SMAT_C_F16, (int32_t)kernel, 0, stream};
        rc = g_launch(vals, row_ptr, col_idx, b, p[4], size[0], size[1], size[2], size[3], &o, plan);
    }
    Py_END_ALLOW_THREADS
    if (rc) return PyObject_CallFunction(g_check, "i", rc); // raises
    Py_RETURN_NONE;
}

// Addresses of the two entry points, the function in Python, what raises for a status, and the class of plans.
PyObject *bind(PyObject *, PyObject *args)
{
    unsigned long long launch, drop_in;
    PyObject *in_python, *check, *plan_type;
    if (!PyArg_ParseTuple(args, "KKOOO", &launch, &drop_in, &in_python, &check, &plan_type)) return nullptr;
    g_launch = reinterpret_cast<decltype(g_launch)>(launch);
    g_launch_drop_in = reinterpret_cast<decltype(g_launch_drop_in)>(drop_in);
    Py_INCREF(in_python);
    Py_INCREF(check);
    Py_INCREF(plan_type);
    Py_XSETREF(g_in_python, in_python);
    Py_XSETREF(g_check, check);
    Py_XSETREF(g_plan_type, plan_type);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"spmm", (PyCFunction)(void (*)(void))spmm, METH_FASTCALL | METH_KEYWORDS,
     "spmm($module, vals, row_ptr, col_idx, B, C_out, M, N, K, nnzb, plan=None, c_f32=False, kernel=0, stream=None, drop_in=False, b_row_major=False)\n--\n\n"
     "Launch the SpMM on device tensors (anything with .data_ptr()).\n\n"
     "drop_in=True calls the positional drop-in entry point (smat_spmm_bcsr_f16) with\nNULL block_info / rel_map; otherwise the options entry point."},
    {"bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__call(void)
{
    g_data_ptr = PyUnicode_InternFromString("data_ptr");
    g_address = PyUnicode_InternFromString("_address");
    if (!g_data_ptr || !g_address) return nullptr;
    for (int i = 0; i < N_ARGS; i++)
        if (!(g_names[i] = PyUnicode_InternFromString(NAMES[i]))) return nullptr;
    return PyModule_Create(&module);
}

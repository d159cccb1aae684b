// The call paths of the Python package in native code: tensors are checked and described, the output is allocated and the
// C ABI is called without going back to the interpreter.  A call costs ~2 us of host time beyond the launch, where the same
// steps in Python and ctypes cost ~10: more than a small decode kernel runs.
//
// Every function here takes the plain case of its operator only -- the types, layouts and options of ordinary calls -- and
// returns None (False) for anything else; the Python implementation then takes the call, converts what it converts and
// raises what it raises.  Nothing is remembered between calls: tensors are described afresh each time, workspaces come from
// the package's own table.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/tilegym_hip.h"

namespace {

decltype(&tg_fp8_gemm) g_gemm = nullptr;
decltype(&tg_fp8_gemm_workspace_bytes) g_gemm_workspace_bytes = nullptr;
decltype(&tg_fp8_ragged_gemm) g_ragged_gemm = nullptr;
decltype(&tg_fp8_quant_group) g_quant_group = nullptr;
decltype(&tg_fp8_fused_moe) g_fused_moe = nullptr;
decltype(&tg_fp8_fused_moe_block_m) g_fused_moe_block_m = nullptr;
decltype(&tg_fp8_fused_moe_workspace_bytes) g_fused_moe_workspace_bytes = nullptr;
PyObject* g_workspaces = nullptr;     // {(device, stream, under capture): [scratch tensors, newest last]}
PyObject* g_workspace_for = nullptr;  // callable(device, bytes, index, stream) -> tensor, for a new or larger one
PyObject* g_check_rc = nullptr;       // callable(rc, where): raises

constexpr int64_t kMaxMoeTokens = 32768;  // one chunk of the layer

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return TG_F32;
        case at::kHalf: return TG_F16;
        case at::kBFloat16: return TG_BF16;
        case at::kInt: return TG_I32;
        case at::kLong: return TG_I64;
        case at::kFloat8_e5m2: return TG_F8E5M2;
        case at::kByte: return 6;  // (workspaces; no operand has this type)
        case at::kFloat8_e4m3fn: return TG_F8E4M3FN;
        case at::kChar: return TG_I8;
        default: return -1;
    }
}

bool describe(const at::Tensor& t, tg_tensor* d) {
    const int code = dtype_code(t.scalar_type());
    const int64_t nd = t.dim();
    if (code < 0 || nd > TG_MAX_DIMS) return false;
    *d = tg_tensor{};
    d->ptr = reinterpret_cast<uint64_t>(t.data_ptr());
    d->ndim = (int32_t)nd;
    d->dtype = code;
    for (int64_t i = 0; i < nd; ++i) {
        d->shape[i] = t.size(i);
        d->strides[i] = t.stride(i);
    }
    return true;
}

tg_tensor describe_rows(const at::Tensor& t, int64_t rows, int64_t cols) {  // a contiguous tensor as (rows, cols)
    tg_tensor d{};
    d.ptr = reinterpret_cast<uint64_t>(t.data_ptr());
    d.ndim = 2;
    d.dtype = dtype_code(t.scalar_type());
    d.shape[0] = rows; d.shape[1] = cols;
    d.strides[0] = cols; d.strides[1] = 1;
    return d;
}

const at::Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

bool on_gpu(const at::Tensor* t) { return t && t->is_cuda() && t->layout() == at::kStrided; }
bool plain(const at::Tensor* t, at::ScalarType type, int64_t dim) {
    return on_gpu(t) && t->scalar_type() == type && t->dim() == dim && t->is_contiguous();
}
bool io_type(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf || t == at::kFloat; }

at::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

// The scratch buffer of the current stream, at least `bytes`, described; false with an exception set.
bool workspace(PyObject* like, int index, hipStream_t stream, int64_t bytes, tg_tensor* d) {
    const bool capturing = c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
    PyObject* key = Py_BuildValue("(iKO)", index, (unsigned long long)(uintptr_t)stream, capturing ? Py_True : Py_False);
    if (!key) return false;
    PyObject* held = PyDict_GetItemWithError(g_workspaces, key);
    Py_DECREF(key);
    if (held && PyList_Check(held) && PyList_GET_SIZE(held) > 0) {
        const at::Tensor* t = tensor_of(PyList_GET_ITEM(held, PyList_GET_SIZE(held) - 1));
        if (t && t->numel() >= bytes) return describe(*t, d);
    } else if (!held && PyErr_Occurred()) {
        return false;
    }
    PyObject* device = PyObject_GetAttrString(like, "device");
    if (!device) return false;
    PyObject* made = PyObject_CallFunction(g_workspace_for, "OLiK", device, (long long)bytes, index, (unsigned long long)(uintptr_t)stream);
    Py_DECREF(device);
    if (!made) return false;
    const at::Tensor* t = tensor_of(made);  // (the table keeps it alive)
    const bool ok = t && describe(*t, d);
    Py_DECREF(made);
    if (!ok && !PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "no workspace");
    return ok;
}

// Raises what check_rc raises for rc != 0; true when rc is 0.
bool succeeded(int32_t rc, const char* where) {
    if (rc == TG_OK) return true;
    PyObject* r = PyObject_CallFunction(g_check_rc, "is", (int)rc, where);
    Py_XDECREF(r);
    if (r) PyErr_SetString(PyExc_RuntimeError, where);
    return false;
}

// None -> no scale; a number -> into alpha; a tensor -> the kernel reads it.  False: not a plain scale.
bool take_scale(PyObject* o, double* alpha, const at::Tensor** t) {
    *t = nullptr;
    if (o == Py_None) return true;
    if (PyFloat_Check(o)) { *alpha *= PyFloat_AS_DOUBLE(o); return true; }
    const at::Tensor* s = tensor_of(o);
    if (!on_gpu(s) || s->scalar_type() != at::kFloat || !s->is_contiguous() || s->dim() > TG_MAX_DIMS) return false;
    *t = s;
    return true;
}

// tg_fp8_gemm on described tensors; false with an exception set.
bool run_gemm(PyObject* like, const at::Tensor& a, const tg_tensor& dc, const tg_tensor& da, const tg_tensor& db, const at::Tensor* sa,
              const at::Tensor* sb, const tg_tensor* dsa, const tg_tensor* dsb, bool trans_a, bool trans_b, double alpha, double beta, bool use_workspace) {
    const int index = a.get_device();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(index).stream();
    tg_tensor tsa, tsb, dws;
    if (!dsa && sa) { if (!describe(*sa, &tsa)) { PyErr_SetString(PyExc_TypeError, "scale_a"); return false; } dsa = &tsa; }
    if (!dsb && sb) { if (!describe(*sb, &tsb)) { PyErr_SetString(PyExc_TypeError, "scale_b"); return false; } dsb = &tsb; }
    const int64_t M = da.shape[trans_a ? 1 : 0], K = da.shape[trans_a ? 0 : 1], N = db.shape[trans_b ? 0 : 1];
    const int64_t need = use_workspace && M > 0 && N > 0 && K > 0 ? g_gemm_workspace_bytes(M, N, K, trans_b, nullptr, 0) : 0;
    if (need > 0 && !workspace(like, index, stream, need, &dws)) return false;
    int32_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_gemm(&dc, &da, &db, dsa, dsb, trans_a, trans_b, (float)alpha, (float)beta, need > 0 ? &dws : nullptr, nullptr, 0, index,
                (uint64_t)(uintptr_t)stream);
    Py_END_ALLOW_THREADS
    return succeeded(rc, "tg_fp8_gemm");
}

// matmul(a, b, trans_a, trans_b, scale_a, scale_b, alpha, out_dtype) -> tensor, or None
PyObject* py_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 8) { PyErr_SetString(PyExc_TypeError, "matmul takes 8 arguments"); return nullptr; }
    const at::Tensor *a = tensor_of(args[0]), *b = tensor_of(args[1]), *sa, *sb;
    if (!plain(a, at::kFloat8_e4m3fn, 2) || !plain(b, at::kFloat8_e4m3fn, 2)) Py_RETURN_NONE;
    const bool trans_a = args[2] == Py_True, trans_b = args[3] == Py_True;
    double alpha = PyFloat_AsDouble(args[6]);
    if (alpha == -1.0 && PyErr_Occurred()) return nullptr;
    if (!take_scale(args[4], &alpha, &sa) || !take_scale(args[5], &alpha, &sb)) Py_RETURN_NONE;
    at::ScalarType out = at::kFloat8_e4m3fn;
    if (args[7] != Py_None) {
        if (!THPDtype_Check(args[7])) Py_RETURN_NONE;
        out = reinterpret_cast<THPDtype*>(args[7])->scalar_type;
        if (!io_type(out) && out != at::kFloat8_e4m3fn) Py_RETURN_NONE;
    }
    const int64_t M = a->size(trans_a ? 1 : 0), K = a->size(trans_a ? 0 : 1), N = b->size(trans_b ? 0 : 1), Kb = b->size(trans_b ? 1 : 0);
    if (K != Kb || a->device() != b->device()) Py_RETURN_NONE;
    at::Tensor c = new_tensor({M, N}, out, *a);
    tg_tensor dc, da, db;
    if (!describe(c, &dc) || !describe(*a, &da) || !describe(*b, &db)) Py_RETURN_NONE;
    if (!run_gemm(args[0], *a, dc, da, db, sa, sb, nullptr, nullptr, trans_a, trans_b, alpha, 0.0, true)) return nullptr;
    return THPVariable_Wrap(std::move(c));
    END_HANDLE_TH_ERRORS
}

// gemm(c, a, b, scale_a, scale_b, trans_a, trans_b, alpha, beta, use_workspace) -> True, or False
PyObject* py_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 10) { PyErr_SetString(PyExc_TypeError, "gemm takes 10 arguments"); return nullptr; }
    const at::Tensor *c = tensor_of(args[0]), *a = tensor_of(args[1]), *b = tensor_of(args[2]);
    const at::Tensor *sa = args[3] == Py_None ? nullptr : tensor_of(args[3]), *sb = args[4] == Py_None ? nullptr : tensor_of(args[4]);
    if (!on_gpu(c) || !on_gpu(a) || !on_gpu(b) || (args[3] != Py_None && !on_gpu(sa)) || (args[4] != Py_None && !on_gpu(sb))) Py_RETURN_FALSE;
    tg_tensor dc, da, db, dsa, dsb;
    if (a->dim() != 2 || b->dim() != 2 || !describe(*c, &dc) || !describe(*a, &da) || !describe(*b, &db) || (sa && !describe(*sa, &dsa)) ||
        (sb && !describe(*sb, &dsb)))
        Py_RETURN_FALSE;
    const double alpha = PyFloat_AsDouble(args[7]), beta = PyFloat_AsDouble(args[8]);
    if (PyErr_Occurred()) return nullptr;
    if (!run_gemm(args[1], *a, dc, da, db, nullptr, nullptr, sa ? &dsa : nullptr, sb ? &dsb : nullptr, args[5] == Py_True, args[6] == Py_True, alpha,
                  beta, args[9] == Py_True))
        return nullptr;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// block_matmul(A, B, As, Bs, out_dtype) -> tensor, or None: 128 x 128 quantization blocks
PyObject* py_block_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) { PyErr_SetString(PyExc_TypeError, "block_matmul takes 5 arguments"); return nullptr; }
    const at::Tensor *a = tensor_of(args[0]), *b = tensor_of(args[1]), *as = tensor_of(args[2]), *bs = tensor_of(args[3]);
    if (!on_gpu(a) || a->dim() < 1 || !plain(a, at::kFloat8_e4m3fn, a->dim()) || !plain(b, at::kFloat8_e4m3fn, 2) || !on_gpu(as) ||
        !plain(as, at::kFloat, a->dim()) || !plain(bs, at::kFloat, 2) || !THPDtype_Check(args[4]))
        Py_RETURN_NONE;
    const at::ScalarType out = reinterpret_cast<THPDtype*>(args[4])->scalar_type;
    const int64_t nd = a->dim(), K = a->size(nd - 1), N = b->size(0), kb = (K + 127) / 128;
    if (!io_type(out) || b->size(1) != K || K == 0 || a->numel() == 0 || as->size(nd - 1) != kb || bs->size(0) != (N + 127) / 128 ||
        bs->size(1) != kb || a->device() != b->device())
        Py_RETURN_NONE;
    c10::SmallVector<int64_t, 4> sizes(a->sizes().begin(), a->sizes().end());
    for (int64_t i = 0; i + 1 < nd; ++i)
        if (as->size(i) != sizes[i]) Py_RETURN_NONE;
    sizes[nd - 1] = N;
    const int64_t M = a->numel() / K;
    at::Tensor c = new_tensor(sizes, out, *a);
    const tg_tensor dc = describe_rows(c, M, N), da = describe_rows(*a, M, K), db = describe_rows(*b, N, K), das = describe_rows(*as, M, kb),
                    dbs = describe_rows(*bs, bs->size(0), kb);
    if (!run_gemm(args[0], *a, dc, da, db, nullptr, nullptr, &das, &dbs, false, true, 1.0, 0.0, true)) return nullptr;
    return THPVariable_Wrap(std::move(c));
    END_HANDLE_TH_ERRORS
}

// act_quant(x, group_size, eps, rule) -> (q e4m3, scales row-major), or None
PyObject* py_act_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) { PyErr_SetString(PyExc_TypeError, "act_quant takes 4 arguments"); return nullptr; }
    const at::Tensor* x = tensor_of(args[0]);
    const long group = PyLong_AsLong(args[1]), rule = PyLong_AsLong(args[3]);
    const double eps = PyFloat_AsDouble(args[2]);
    if (PyErr_Occurred()) return nullptr;
    if (!on_gpu(x) || !io_type(x->scalar_type()) || !x->is_contiguous() || x->dim() < 1 || x->dim() > TG_MAX_DIMS || group <= 0 ||
        x->size(x->dim() - 1) % group != 0)
        Py_RETURN_NONE;
    at::Tensor q = new_tensor(x->sizes(), at::kFloat8_e4m3fn, *x);
    c10::SmallVector<int64_t, 4> sizes(x->sizes().begin(), x->sizes().end());
    sizes.back() /= group;
    at::Tensor scales = new_tensor(sizes, at::kFloat, *x);
    tg_tensor dq, ds, dx;
    if (!describe(q, &dq) || !describe(scales, &ds) || !describe(*x, &dx)) Py_RETURN_NONE;
    const int index = x->get_device();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(index).stream();
    int32_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_quant_group(&dq, &ds, &dx, (int32_t)group, (float)eps, (int32_t)rule, index, (uint64_t)(uintptr_t)stream);
    Py_END_ALLOW_THREADS
    if (!succeeded(rc, "tg_fp8_quant_group")) return nullptr;
    PyObject* tuple = PyTuple_New(2);
    if (!tuple) return nullptr;
    PyTuple_SET_ITEM(tuple, 0, THPVariable_Wrap(std::move(q)));
    PyTuple_SET_ITEM(tuple, 1, THPVariable_Wrap(std::move(scales)));
    return tuple;
    END_HANDLE_TH_ERRORS
}

// ragged_matmul(a, b, a_scale, b_scale, m_indptr, out_dtype) -> tensor, or None: 128 x 128 quantization blocks
PyObject* py_ragged_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 6) { PyErr_SetString(PyExc_TypeError, "ragged_matmul takes 6 arguments"); return nullptr; }
    const at::Tensor *a = tensor_of(args[0]), *b = tensor_of(args[1]), *as = tensor_of(args[2]), *bs = tensor_of(args[3]), *ptr = tensor_of(args[4]);
    if (!plain(a, at::kFloat8_e4m3fn, 2) || !plain(b, at::kFloat8_e4m3fn, 3) || !plain(as, at::kFloat, 2) || !plain(bs, at::kFloat, 3) ||
        !plain(ptr, at::kInt, 1))
        Py_RETURN_NONE;
    at::ScalarType out = at::kBFloat16;
    if (args[5] != Py_None) {
        if (!THPDtype_Check(args[5])) Py_RETURN_NONE;
        out = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
    }
    const int64_t M = a->size(0), K = a->size(1), E = b->size(0), N = b->size(1), kb = (K + 127) / 128;
    if (!io_type(out) || b->size(2) != K || ptr->size(0) != E + 1 || bs->size(0) != E || bs->size(1) != (N + 127) / 128 || bs->size(2) != kb ||
        as->size(0) != M || as->size(1) != kb || a->device() != b->device())
        Py_RETURN_NONE;
    at::Tensor c = new_tensor({M, N}, out, *a);
    tg_tensor dc, da, db, das, dbs, dptr;
    if (!describe(c, &dc) || !describe(*a, &da) || !describe(*b, &db) || !describe(*as, &das) || !describe(*bs, &dbs) || !describe(*ptr, &dptr))
        Py_RETURN_NONE;
    const int index = a->get_device();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(index).stream();
    int32_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_ragged_gemm(&dc, &da, &db, &das, &dbs, &dptr, nullptr, 0, index, (uint64_t)(uintptr_t)stream);
    Py_END_ALLOW_THREADS
    if (!succeeded(rc, "tg_fp8_ragged_gemm")) return nullptr;
    return THPVariable_Wrap(std::move(c));
    END_HANDLE_TH_ERRORS
}

// fused_moe(hidden, w1, w2, topk_weights, topk_ids, w1_scale, w2_scale, inplace, max_experts) -> tensor, or None: the whole layer
// when tg_fp8_fused_moe takes it as one chunk
PyObject* py_fused_moe(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 9) { PyErr_SetString(PyExc_TypeError, "fused_moe takes 9 arguments"); return nullptr; }
    const at::Tensor *x = tensor_of(args[0]), *w1 = tensor_of(args[1]), *w2 = tensor_of(args[2]), *tw = tensor_of(args[3]), *ids = tensor_of(args[4]),
                     *s1 = tensor_of(args[5]), *s2 = tensor_of(args[6]);
    const long max_experts = PyLong_AsLong(args[8]);
    if (PyErr_Occurred()) return nullptr;
    if (!on_gpu(x) || (x->scalar_type() != at::kBFloat16 && x->scalar_type() != at::kHalf) || x->dim() != 2 || !x->is_contiguous() ||
        !plain(w1, at::kFloat8_e4m3fn, 3) || !plain(w2, at::kFloat8_e4m3fn, 3) || !plain(tw, at::kFloat, 2) || !on_gpu(ids) ||
        (ids->scalar_type() != at::kInt && ids->scalar_type() != at::kLong) || ids->dim() != 2 || !ids->is_contiguous() || !plain(s1, at::kFloat, 3) ||
        !plain(s2, at::kFloat, 3))
        Py_RETURN_NONE;
    const int64_t T = x->size(0), H = x->size(1), E = w1->size(0), I2 = w1->size(1), k = ids->size(1);
    if (T < 1 || T > kMaxMoeTokens || E < 1 || E > max_experts || k < 1 || H % 128 != 0 || H < 128 || H > 65536 || I2 % 256 != 0 || I2 == 0 ||
        w1->size(2) != H || w2->size(0) != E || w2->size(1) != H || w2->size(2) != I2 / 2 || ids->size(0) != T || tw->sizes() != ids->sizes() ||
        x->device() != w1->device() || x->device() != w2->device())
        Py_RETURN_NONE;
    const int block_m = g_fused_moe_block_m(T, k, E, I2 / 2);
    const bool inplace = args[7] == Py_True;
    at::Tensor out = inplace ? *x : new_tensor({T, H}, x->scalar_type(), *x);
    tg_tensor dout, dx, dw1, dw2, ds1, ds2, dtw, dids, dws;
    if (!describe(out, &dout) || !describe(*x, &dx) || !describe(*w1, &dw1) || !describe(*w2, &dw2) || !describe(*s1, &ds1) || !describe(*s2, &ds2) ||
        !describe(*tw, &dtw) || !describe(*ids, &dids))
        Py_RETURN_NONE;
    const int index = x->get_device();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(index).stream();
    if (!workspace(args[0], index, stream, g_fused_moe_workspace_bytes(T, k, E, H, I2 / 2, block_m), &dws)) return nullptr;
    int32_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_fused_moe(&dout, &dx, &dw1, &dw2, &ds1, &ds2, &dtw, &dids, &dws, block_m, index, (uint64_t)(uintptr_t)stream);
    Py_END_ALLOW_THREADS
    if (!succeeded(rc, "tg_fp8_fused_moe")) return nullptr;
    if (inplace) {
        Py_INCREF(args[0]);
        return args[0];
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// set_up({name: address}, workspaces, workspace_for, check_rc)
PyObject* py_set_up(PyObject*, PyObject* args) {
    PyObject *table, *workspaces, *workspace_for, *check_rc;
    if (!PyArg_ParseTuple(args, "O!O!OO", &PyDict_Type, &table, &PyDict_Type, &workspaces, &workspace_for, &check_rc)) return nullptr;
    auto find = [&](const char* name, auto* slot) {
        PyObject* o = PyDict_GetItemString(table, name);
        const unsigned long long address = o ? PyLong_AsUnsignedLongLong(o) : 0;
        if (!address && !PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "no address for %s", name);
        *slot = reinterpret_cast<std::remove_pointer_t<decltype(slot)>>((uintptr_t)address);
        return !PyErr_Occurred();
    };
    if (!find("tg_fp8_gemm", &g_gemm) || !find("tg_fp8_gemm_workspace_bytes", &g_gemm_workspace_bytes) || !find("tg_fp8_ragged_gemm", &g_ragged_gemm) ||
        !find("tg_fp8_quant_group", &g_quant_group) || !find("tg_fp8_fused_moe", &g_fused_moe) ||
        !find("tg_fp8_fused_moe_block_m", &g_fused_moe_block_m) || !find("tg_fp8_fused_moe_workspace_bytes", &g_fused_moe_workspace_bytes))
        return nullptr;
    for (auto [slot, o] : {std::pair{&g_workspaces, workspaces}, std::pair{&g_workspace_for, workspace_for}, std::pair{&g_check_rc, check_rc}}) {
        Py_INCREF(o);
        Py_XDECREF(*slot);
        *slot = o;
    }
    Py_RETURN_NONE;
}

#define TG_FAST(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {TG_FAST("matmul", py_matmul),
                          TG_FAST("gemm", py_gemm),
                          TG_FAST("block_matmul", py_block_matmul),
                          TG_FAST("act_quant", py_act_quant),
                          TG_FAST("ragged_matmul", py_ragged_matmul),
                          TG_FAST("fused_moe", py_fused_moe),
                          {"set_up", py_set_up, METH_VARARGS, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&kModule); }

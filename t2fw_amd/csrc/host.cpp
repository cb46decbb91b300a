// The host side of a call, from torch tensors to the C ABI (include/t2fw_hip.h): checks, allocations and the launch in one
// step.  The same through ctypes costs a Python operation per shape, type, pointer and output.  What the calls mean,
// which kernels they ask for and what is an error stays in functional_lfw.py and functional_dfw.py.
//
// Host time of a call, 4 x 16 tokens of 64 x 64 fp16, ctypes / this: forward 29.5 / 19.1 us without gradients, a training step
// 205 / 152 us (of which torch's own hand-over to a Python autograd function and back is 91), one generation step 14.6 / 8.4.
// Gates, event and block copies with their results in the same step as the launch: a training step on gate logits (8 x 1000 tokens, 12
// heads, bf16) 181 / 168, of 128-wide heads (24 x 1024, fp16) 260 / 219.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>

#include <vector>

#include "../../include/t2fw_hip.h"

namespace {

using at::Tensor;

const Tensor &tensor(PyObject *o) {
    TORCH_CHECK(THPVariable_Check(o), "t2fw: expected a tensor");
    return THPVariable_Unpack(o);
}
int64_t integer(PyObject *o) {
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}
void *address(PyObject *o) {
    void *v = PyLong_AsVoidPtr(o);
    if (v == nullptr && PyErr_Occurred()) throw python_error();
    return v;
}
void arguments(Py_ssize_t n, Py_ssize_t want) { TORCH_CHECK(n == want, "t2fw: ", n, " arguments, expected ", want); }
void done(int rc) {
    TORCH_CHECK_WITH(Error, rc == 0, "t2fw error ", rc, ": ", t2fw_last_error());
}
PyObject *wrapped(std::initializer_list<Tensor> ts) {
    PyObject *t = PyTuple_New((Py_ssize_t)ts.size());
    if (t == nullptr) throw python_error();
    Py_ssize_t i = 0;
    for (const Tensor &v : ts) {
        PyObject *o = v.defined() ? THPVariable_Wrap(v) : Py_NewRef(Py_None);
        if (o == nullptr) {
            Py_DECREF(t);
            throw python_error();
        }
        PyTuple_SET_ITEM(t, i++, o);
    }
    return t;
}
// The launches run without the interpreter's lock: they wait where the device's queue is full.
template <typename F> int unlocked(F &&launch) {
    pybind11::gil_scoped_release release;
    return launch();
}
// torch.empty_like: a tensor subclass has its own
Tensor empty_like(PyObject *o) {
    if (THPVariable_CheckExact(o)) return at::empty_like(tensor(o));
    const pybind11::object made = pybind11::module_::import("torch").attr("empty_like")(pybind11::handle(o));
    return tensor(made.ptr());
}
Tensor bytes_like(const Tensor &t, int64_t n) { return at::empty({n}, t.options().dtype(at::kByte)); }

// lfw_shape(x, f, q, k, f_key, state, heads) -> (B, T, H, D, K), or None where a call on these is an error
PyObject *lfw_shape(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 7);
    for (int i = 0; i < 6; ++i)
        if (!THPVariable_Check(a[i])) Py_RETURN_NONE;
    const Tensor &x = tensor(a[0]), &q = tensor(a[2]), &s = tensor(a[5]);
    const int64_t lead = a[6] == Py_True ? 3 : 2;
    for (int i = 0; i < 6; ++i) {
        const Tensor &t = tensor(a[i]);
        if (!t.is_cuda() || !t.is_contiguous() || t.dim() != lead + 1 || t.scalar_type() != x.scalar_type()) Py_RETURN_NONE;
    }
    if (tensor(a[1]).sizes() != x.sizes() || tensor(a[3]).sizes() != q.sizes() || tensor(a[4]).sizes() != q.sizes()) Py_RETURN_NONE;
    const int64_t B = x.size(0), T = x.size(1), H = lead == 3 ? x.size(2) : 1, D = x.size(lead), K = q.size(lead);
    if (q.size(0) != B || q.size(1) != T || (lead == 3 && q.size(2) != H)) Py_RETURN_NONE;
    if (s.size(0) != B || (lead == 3 && s.size(1) != H) || s.size(lead - 1) != D || s.size(lead) != K) Py_RETURN_NONE;
    return Py_BuildValue("(LLLLL)", (long long)B, (long long)T, (long long)H, (long long)D, (long long)K);
    END_HANDLE_TH_ERRORS
}

// lfw_forward(x, f, q, k, f_key, state, heads, checkpoints per row or -1 for none, C, dtype, flags, workspace address or 0, its bytes,
// stream, logits, event or 0) -> (outputs, next_state, checkpoints or None); address 0: the workspace is allocated for the call;
// logits: f and f_key are gate logits, and the gates follow in the result; event: recorded after the launch
PyObject *lfw_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 16);
    const Tensor &x = tensor(a[0]), &q = tensor(a[2]), &k = tensor(a[3]), &s = tensor(a[5]);
    const bool heads = a[6] == Py_True, logits = a[14] == Py_True;
    const Tensor &lf = tensor(a[1]), &lk = tensor(a[4]);
    Tensor made_f, made_fk;
    if (logits) {
        made_f = empty_like(a[1]);
        made_fk = empty_like(a[4]);
    }
    const Tensor &f = logits ? made_f : lf, &fk = logits ? made_fk : lk;
    void *const event = address(a[15]);
    const int64_t nc = integer(a[7]), ws_bytes = integer(a[12]);
    const int32_t C = (int32_t)integer(a[8]), dtype = (int32_t)integer(a[9]), flags = (int32_t)integer(a[10]);
    void *ws = address(a[11]), *const stream = address(a[13]);
    const int64_t B = x.size(0), T = x.size(1), H = heads ? x.size(2) : 1, D = x.size(-1), K = q.size(-1);
    const Tensor out = empty_like(a[0]), next = empty_like(a[5]);
    Tensor ckpt, scratch;
    if (nc >= 0) ckpt = at::empty({B * H, nc, D, K}, x.options());
    if (ws == nullptr && ws_bytes > 0) {
        scratch = bytes_like(x, ws_bytes);
        ws = scratch.data_ptr();
    }
    void *const ck = ckpt.defined() ? ckpt.data_ptr() : nullptr;
    // whether the chunks of a row run side by side depends on the call (its rows, with or without gradients), and the bits with it
    size_t extra = at::globalContext().deterministicAlgorithms() ? 0 : t2fw_lfw_forward_scratch_bytes(B, T, H, D, K, C, dtype, flags, ckpt.defined());
    Tensor chunks;
    if (extra > 0) {
        try {
            chunks = bytes_like(x, (int64_t)extra);
        } catch (const c10::OutOfMemoryError &) {        // up to 420 MB, which the sequential kernel does without
            extra = 0;
        }
    }
    done(unlocked([&] {
        if (logits) {
            const int rc = t2fw_gate_forward(lf.data_ptr(), lk.data_ptr(), f.data_ptr(), fk.data_ptr(), lf.numel(), lk.numel(), dtype, stream);
            if (rc) return rc;
        }
        const int rc = extra > 0 ? t2fw_lfw_forward_scratch(x.data_ptr(), f.data_ptr(), q.data_ptr(), k.data_ptr(), fk.data_ptr(), s.data_ptr(),
                                                            out.data_ptr(), next.data_ptr(), ck, B, T, H, D, K, C, dtype, flags, ws, ws_bytes,
                                                            chunks.data_ptr(), extra, stream)
                     : heads ? t2fw_lfw_forward_heads(x.data_ptr(), f.data_ptr(), q.data_ptr(), k.data_ptr(), fk.data_ptr(), s.data_ptr(),
                                              out.data_ptr(), next.data_ptr(), ck, B, T, H, D, K, C, dtype, flags, ws, ws_bytes, stream)
                     : t2fw_lfw_forward(x.data_ptr(), f.data_ptr(), q.data_ptr(), k.data_ptr(), fk.data_ptr(), s.data_ptr(),
                                        out.data_ptr(), next.data_ptr(), ck, B, T, D, K, C, dtype, flags, ws, ws_bytes, stream);
        return rc || event == nullptr ? rc : t2fw_record_event(event, stream);
    }));
    return logits ? wrapped({out, next, ckpt, f, fk}) : wrapped({out, next, ckpt});
    END_HANDLE_TH_ERRORS
}

// lfw_backward_arguments(g_out, g_state, x, f, q, k, f_key, state, checkpoints, heads, C, dtype, flags, workspace bytes, stream)
// -> ((d_x, d_f, d_q, d_k, d_f_key, d_state), arguments of t2fw_lfw_backward or t2fw_lfw_backward_heads, workspace or None).
// The call itself is Python's: which kernels it asks for can be seen there.
PyObject *lfw_backward_arguments(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 15);
    const bool heads = a[9] == Py_True;
    const Tensor &x = tensor(a[2]), &q = tensor(a[4]);
    const int64_t ws_bytes = integer(a[13]);
    Tensor grads[6], scratch;
    for (int i = 0; i < 6; ++i) grads[i] = empty_like(a[2 + i]);
    if (ws_bytes > 0) scratch = bytes_like(x, ws_bytes);
    std::vector<long long> v;                      // addresses, sizes and options in the order of the C declaration
    v.reserve(25);
    for (int i = 0; i < 9; ++i) v.push_back((long long)(uintptr_t)tensor(a[i]).data_ptr());
    for (const Tensor &g : grads) v.push_back((long long)(uintptr_t)g.data_ptr());
    v.push_back(x.size(0));
    v.push_back(x.size(1));
    if (heads) v.push_back(x.size(2));
    v.push_back(x.size(-1));
    v.push_back(q.size(-1));
    for (int i = 10; i < 13; ++i) v.push_back(integer(a[i]));
    v.push_back(scratch.defined() ? (long long)(uintptr_t)scratch.data_ptr() : 0);
    v.push_back(ws_bytes);
    v.push_back((long long)(uintptr_t)address(a[14]));
    pybind11::tuple args(v.size());
    for (size_t i = 0; i < v.size(); ++i) {
        PyObject *o = PyLong_FromLongLong(v[i]);
        if (o == nullptr) throw python_error();
        PyTuple_SET_ITEM(args.ptr(), (Py_ssize_t)i, o);
    }
    pybind11::object g = pybind11::reinterpret_steal<pybind11::object>(wrapped({grads[0], grads[1], grads[2], grads[3], grads[4], grads[5]}));
    pybind11::object w = pybind11::reinterpret_steal<pybind11::object>(scratch.defined() ? THPVariable_Wrap(scratch) : Py_NewRef(Py_None));
    return PyTuple_Pack(3, g.ptr(), args.ptr(), w.ptr());
    END_HANDLE_TH_ERRORS
}

// lfw_step(x, f, q, k, f_key, state, out or None, inplace, stream) -> (out, state), or None where it is an error
PyObject *lfw_step(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 9);
    for (int i = 0; i < 6; ++i)
        if (!THPVariable_Check(a[i])) Py_RETURN_NONE;
    const Tensor &x = tensor(a[0]), &f = tensor(a[1]), &q = tensor(a[2]), &k = tensor(a[3]), &fk = tensor(a[4]), &s = tensor(a[5]);
    for (int i = 0; i < 6; ++i) {
        const Tensor &t = tensor(a[i]);
        if (!t.is_cuda() || !t.is_contiguous() || t.dim() != (i == 5 ? 3 : 2) || t.scalar_type() != x.scalar_type()) Py_RETURN_NONE;
    }
    const int64_t B = x.size(0), D = x.size(1), K = q.size(1);
    if (f.sizes() != x.sizes() || k.sizes() != q.sizes() || fk.sizes() != q.sizes() || q.size(0) != B || s.size(0) != B ||
        s.size(1) != D || s.size(2) != K)
        Py_RETURN_NONE;
    int32_t dtype;
    switch (x.scalar_type()) {
        case at::kFloat: dtype = T2FW_F32; break;
        case at::kHalf: dtype = T2FW_F16; break;
        case at::kBFloat16: dtype = T2FW_BF16; break;
        case at::kDouble: dtype = T2FW_F64; break;
        default: Py_RETURN_NONE;
    }
    void *const stream = address(a[8]);
    const Tensor out = a[6] == Py_None ? empty_like(a[0]) : tensor(a[6]), next = a[7] == Py_True ? s : empty_like(a[5]);
    done(unlocked([&] {
        return t2fw_lfw_step(x.data_ptr(), f.data_ptr(), q.data_ptr(), k.data_ptr(), fk.data_ptr(), s.data_ptr(), out.data_ptr(),
                             next.data_ptr(), B, D, K, dtype, stream);
    }));
    return wrapped({out, next});
    END_HANDLE_TH_ERRORS
}

// dfw_forward(q, k, v, state, dtype, flags, stream) -> (outputs, final_state, delta)
PyObject *dfw_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 7);
    const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &s = tensor(a[3]);
    const int32_t dtype = (int32_t)integer(a[4]), flags = (int32_t)integer(a[5]);
    void *const stream = address(a[6]);
    const Tensor out = empty_like(a[2]), fin = empty_like(a[3]), delta = empty_like(a[2]);
    done(unlocked([&] {
        return t2fw_dfw_forward(q.data_ptr(), k.data_ptr(), v.data_ptr(), s.data_ptr(), out.data_ptr(), fin.data_ptr(), delta.data_ptr(),
                                v.size(0), v.size(1), v.size(2), q.size(2), dtype, flags, stream);
    }));
    return wrapped({out, fin, delta});
    END_HANDLE_TH_ERRORS
}

// dfw_backward(g_out, g_state, q, k, delta, final_state, dtype, flags, stream) -> (d_q, d_k, d_v, d_state)
PyObject *dfw_backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 9);
    const Tensor &go = tensor(a[0]), &gs = tensor(a[1]), &q = tensor(a[2]), &k = tensor(a[3]), &delta = tensor(a[4]), &fin = tensor(a[5]);
    const int32_t dtype = (int32_t)integer(a[6]), flags = (int32_t)integer(a[7]);
    void *const stream = address(a[8]);
    const Tensor dq = empty_like(a[2]), dk = empty_like(a[3]), dv = empty_like(a[4]), ds = empty_like(a[5]);
    done(unlocked([&] {
        return t2fw_dfw_backward(go.data_ptr(), gs.data_ptr(), q.data_ptr(), k.data_ptr(), delta.data_ptr(), fin.data_ptr(), dq.data_ptr(),
                                 dk.data_ptr(), dv.data_ptr(), ds.data_ptr(), delta.size(0), delta.size(1), delta.size(2), q.size(2),
                                 dtype, flags, stream);
    }));
    return wrapped({dq, dk, dv, ds});
    END_HANDLE_TH_ERRORS
}

// The value blocks' entry points take 16-byte aligned arrays
bool aligned(std::initializer_list<Tensor> ts) {
    for (const Tensor &t : ts)
        if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) return false;
    return true;
}

// dfw_forward_blocks(q, k, v, state, dtype, flags, stream, plan of the copies of q and k or None) -> (outputs, final_state, delta,
// q's copy or None, k's), or None for arrays that t2fw_dfw_forward_blocks does not take (empty, misaligned, very large)
PyObject *dfw_forward_blocks(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 8);
    const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &s = tensor(a[3]);
    const int32_t dtype = (int32_t)integer(a[4]), flags = (int32_t)integer(a[5]);
    void *const stream = address(a[6]);
    const int64_t B = v.size(0), T = v.size(1), D = v.size(2);
    if (B == 0 || T == 0 || T * D >= 0x7fffffffLL || B * (D / 64) > 0x1fffffffLL || !aligned({q, k, v, s})) Py_RETURN_NONE;
    const Tensor out = empty_like(a[2]), fin = empty_like(a[3]), delta = empty_like(a[2]);
    Tensor qc, kc;
    t2fw_block_copy_desc d[2];
    if (a[7] != Py_None) {
        char *plan = nullptr;
        Py_ssize_t len = 0;
        if (PyBytes_AsStringAndSize(a[7], &plan, &len) != 0) throw python_error();
        TORCH_CHECK(len == (Py_ssize_t)sizeof(d), "t2fw: a plan of ", len, " bytes for 2 arrays");
        memcpy(d, plan, sizeof(d));
        qc = empty_like(a[0]);
        kc = empty_like(a[1]);
        d[0].src = q.data_ptr(); d[0].dst = qc.data_ptr();
        d[1].src = k.data_ptr(); d[1].dst = kc.data_ptr();
    }
    done(unlocked([&] {
        const int rc = t2fw_dfw_forward_blocks(q.data_ptr(), k.data_ptr(), v.data_ptr(), s.data_ptr(), out.data_ptr(), fin.data_ptr(),
                                               delta.data_ptr(), B, T, D, q.size(2), dtype, flags, stream);
        return rc || !qc.defined() ? rc : t2fw_block_copy(d, 2, dtype, stream);
    }));
    return wrapped({out, fin, delta, qc, kc});
    END_HANDLE_TH_ERRORS
}

// dfw_backward_blocks(g_out, g_state, q, k, delta, final_state, dtype, flags, stream) -> (d_q, d_k, d_v, d_state); d_q and d_k
// [B, n, T, 64], per block, where t2fw_dfw_backward_sums does not take the call
PyObject *dfw_backward_blocks(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 9);
    Tensor in[6];                                  // gradients, and what a caller's hooks give back, may lie anywhere
    for (int i = 0; i < 6; ++i) in[i] = aligned({tensor(a[i])}) ? tensor(a[i]) : tensor(a[i]).clone();
    const Tensor &go = in[0], &gs = in[1], &q = in[2], &k = in[3], &delta = in[4], &fin = in[5];
    const int32_t dtype = (int32_t)integer(a[6]), flags = (int32_t)integer(a[7]);
    void *const stream = address(a[8]);
    const int64_t B = delta.size(0), T = delta.size(1), D = delta.size(2);
    const Tensor dv = empty_like(a[4]), ds = empty_like(a[5]);
    const size_t ws_bytes = t2fw_dfw_backward_sums_workspace_bytes(B, T, D, q.size(2), dtype, flags);
    if (ws_bytes > 0) {
        const Tensor dq = empty_like(a[2]), dk = empty_like(a[3]), scratch = bytes_like(delta, (int64_t)ws_bytes);
        done(unlocked([&] {
            return t2fw_dfw_backward_sums(go.data_ptr(), gs.data_ptr(), q.data_ptr(), k.data_ptr(), delta.data_ptr(), fin.data_ptr(),
                                            dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ds.data_ptr(), B, T, D, q.size(2), dtype, flags,
                                            scratch.data_ptr(), ws_bytes, stream);
        }));
        return wrapped({dq, dk, dv, ds});
    }
    const Tensor dq = at::empty({B, D / 64, T, 64}, q.options()), dk = at::empty({B, D / 64, T, 64}, k.options());
    done(unlocked([&] {
        return t2fw_dfw_backward_blocks(go.data_ptr(), gs.data_ptr(), q.data_ptr(), k.data_ptr(), delta.data_ptr(), fin.data_ptr(),
                                        dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ds.data_ptr(), B, T, D, q.size(2), dtype, flags, stream);
    }));
    return wrapped({dq, dk, dv, ds});
    END_HANDLE_TH_ERRORS
}

// gate_forward(f_logit, fk_logit, f or None, f_key or None, dtype, stream) -> (f, f_key)
PyObject *gate_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 6);
    const Tensor &lf = tensor(a[0]), &lk = tensor(a[1]);
    const Tensor f = a[2] == Py_None ? empty_like(a[0]) : tensor(a[2]), fk = a[3] == Py_None ? empty_like(a[1]) : tensor(a[3]);
    const int32_t dtype = (int32_t)integer(a[4]);
    void *const stream = address(a[5]);
    done(unlocked([&] {
        return t2fw_gate_forward(lf.data_ptr(), lk.data_ptr(), f.data_ptr(), fk.data_ptr(), lf.numel(), lk.numel(), dtype, stream);
    }));
    return wrapped({f, fk});
    END_HANDLE_TH_ERRORS
}

// gate_backward(d_f, d_f_key, f, f_key, dtype, stream): in place on the first two
PyObject *gate_backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 6);
    const Tensor &df = tensor(a[0]), &dfk = tensor(a[1]), &f = tensor(a[2]), &fk = tensor(a[3]);
    const int32_t dtype = (int32_t)integer(a[4]);
    void *const stream = address(a[5]);
    done(unlocked([&] {
        return t2fw_gate_backward(df.data_ptr(), dfk.data_ptr(), f.data_ptr(), fk.data_ptr(), df.data_ptr(), dfk.data_ptr(), df.numel(),
                                  dfk.numel(), dtype, stream);
    }));
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// block_copy(plan, sources, destinations, dtype, stream): plan is the bytes of the descriptors without their addresses
PyObject *block_copy(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 5);
    char *plan = nullptr;
    Py_ssize_t len = 0;
    if (PyBytes_AsStringAndSize(a[0], &plan, &len) != 0) throw python_error();
    const Py_ssize_t count = PySequence_Size(a[1]);
    TORCH_CHECK(count > 0 && count <= T2FW_BLOCK_COPY_MAX && PySequence_Size(a[2]) == count &&
                    len == count * (Py_ssize_t)sizeof(t2fw_block_copy_desc), "t2fw: a plan of ", len, " bytes for ", count, " arrays");
    t2fw_block_copy_desc d[T2FW_BLOCK_COPY_MAX];
    memcpy(d, plan, (size_t)len);
    for (Py_ssize_t i = 0; i < count; ++i) {
        pybind11::object src = pybind11::reinterpret_steal<pybind11::object>(PySequence_GetItem(a[1], i));
        pybind11::object dst = pybind11::reinterpret_steal<pybind11::object>(PySequence_GetItem(a[2], i));
        if (!src || !dst) throw python_error();
        d[i].src = tensor(src.ptr()).data_ptr();
        d[i].dst = tensor(dst.ptr()).data_ptr();
    }
    const int32_t dtype = (int32_t)integer(a[3]);
    void *const stream = address(a[4]);
    done(unlocked([&] { return t2fw_block_copy(d, (int32_t)count, dtype, stream); }));
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// blocks_of(plan or None, sources, shapes of the results, copied, dtype, stream) -> the results, one after the other: new tensors
// that one launch of t2fw_block_copy fills where `copied` says so, views of their sources elsewhere.  None for a tensor subclass.
PyObject *blocks_of(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arguments(n, 6);
    for (int i = 1; i < 4; ++i) TORCH_CHECK(PyTuple_Check(a[i]), "t2fw: expected a tuple");
    const Py_ssize_t count = PyTuple_GET_SIZE(a[1]);
    TORCH_CHECK(count <= T2FW_BLOCK_COPY_MAX && PyTuple_GET_SIZE(a[2]) == count && PyTuple_GET_SIZE(a[3]) == count, "t2fw: ", count, " arrays");
    for (Py_ssize_t i = 0; i < count; ++i)
        if (!THPVariable_CheckExact(PyTuple_GET_ITEM(a[1], i))) Py_RETURN_NONE;
    t2fw_block_copy_desc d[T2FW_BLOCK_COPY_MAX];
    int32_t copies = 0;
    for (Py_ssize_t i = 0; i < count; ++i) copies += PyTuple_GET_ITEM(a[3], i) == Py_True;
    if (copies > 0) {
        char *plan = nullptr;
        Py_ssize_t len = 0;
        if (PyBytes_AsStringAndSize(a[0], &plan, &len) != 0) throw python_error();
        TORCH_CHECK(len == copies * (Py_ssize_t)sizeof(t2fw_block_copy_desc), "t2fw: a plan of ", len, " bytes for ", copies, " arrays");
        memcpy(d, plan, (size_t)len);
    }
    Tensor out[T2FW_BLOCK_COPY_MAX];
    int32_t c = 0;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject *const shape = PyTuple_GET_ITEM(a[2], i);
        TORCH_CHECK(PyTuple_Check(shape) && PyTuple_GET_SIZE(shape) <= 8, "t2fw: expected a shape");
        const Py_ssize_t nd = PyTuple_GET_SIZE(shape);
        int64_t size[8];
        for (Py_ssize_t m = 0; m < nd; ++m) size[m] = integer(PyTuple_GET_ITEM(shape, m));
        const at::IntArrayRef sizes(size, (size_t)nd);
        const Tensor &src = tensor(PyTuple_GET_ITEM(a[1], i));
        if (PyTuple_GET_ITEM(a[3], i) == Py_True) {
            out[i] = at::empty(sizes, src.options());
            d[c].src = src.data_ptr();
            d[c++].dst = out[i].data_ptr();
        } else {
            out[i] = src.view(sizes);
        }
    }
    const int32_t dtype = (int32_t)integer(a[4]);
    void *const stream = address(a[5]);
    if (copies > 0) done(unlocked([&] { return t2fw_block_copy(d, copies, dtype, stream); }));
    PyObject *const t = PyTuple_New(count);
    if (t == nullptr) throw python_error();
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject *const o = THPVariable_Wrap(out[i]);
        if (o == nullptr) {
            Py_DECREF(t);
            throw python_error();
        }
        PyTuple_SET_ITEM(t, i, o);
    }
    return t;
    END_HANDLE_TH_ERRORS
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(lfw_shape), METHOD(lfw_forward), METHOD(lfw_backward_arguments), METHOD(dfw_forward), METHOD(dfw_backward),
                         METHOD(lfw_step),
                         METHOD(dfw_forward_blocks), METHOD(dfw_backward_blocks),
                         METHOD(gate_forward), METHOD(gate_backward), METHOD(block_copy), METHOD(blocks_of), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_t2fw_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__t2fw_host() { return PyModule_Create(&module); }

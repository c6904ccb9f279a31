// The library calls of an attention layer, and of the fp32 quantiser, from Python without Python: rotary embedding,
// attention of one token, quantising of new tokens.  On few sequences a step is over on the device in 10 to 20 us,
// and the checks, views, allocations and argument conversions of the Python functions took twice that on the host
// (1 x 32 heads x 603 tokens with its rotary embedding: 38.2 us per step in Python, now 13.1, as long as the device is busy with it).
//
// Each function here takes exactly the arguments that need nothing done to them first (plain device tensors
// of one current device, of the right shapes, dtypes and layouts, a workspace that is large enough) and
// returns None for all others: the Python function that called it then goes its own way, with its own
// conversions and error messages.  A number is the library's return code.
#include <algorithm>

#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <ATen/ops/empty_cuda_dispatch.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>

#include "../../include/adkv_hip.h"

namespace {

PyObject *raw_stream = nullptr; // device index -> the current stream as a number

// An ordinary tensor of an ordinary device: no subclass, no transform, no pending negation, no other backend.
const at::Tensor *plain(PyObject *o)
{
    static const c10::DispatchKeySet allowed =
        c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) |
        c10::getAutogradRelatedKeySetFromBackend(c10::BackendComponent::CUDABit) |
        c10::getAutocastRelatedKeySetFromBackend(c10::BackendComponent::CUDABit);
    if (!THPVariable_CheckExact(o))
        return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && (t.key_set() | allowed) == allowed ? &t : nullptr;
}

// Nothing watches or transforms what this thread does with tensors: no mode, no tracer, no functorch layer.
bool unwatched()
{
    static const c10::DispatchKeySet ordinary = c10::default_included_set |
                                                c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) |
                                                c10::DispatchKeySet(c10::DispatchKey::BackendSelect);
    return (c10::impl::tls_local_dispatch_key_set().included_ | ordinary) == ordinary && !at::impl::torch_function_mode_enabled();
}

bool half_type(const at::Tensor &t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }

// whether `device` is the thread's current one; its current stream
bool current(c10::Device device, void *&stream)
{
    if (c10::impl::getDeviceGuardImpl(c10::DeviceType::CUDA)->getDevice() != device)
        return false;
    PyObject *i = PyLong_FromLong(device.index());
    PyObject *s = i ? PyObject_CallOneArg(raw_stream, i) : nullptr;
    Py_XDECREF(i);
    if (!s) {
        PyErr_Clear();
        return false;
    }
    stream = PyLong_AsVoidPtr(s);
    Py_DECREF(s);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

// at::empty where its dispatch ends for an ordinary thread (unwatched), on like's device; through the dispatcher while a profiler
// or another observer of operators is on, which is told of them there.  The host's part of a step of 1 x 32 heads x 603 tokens with
// its rotary embedding, four tensors: 14.4 us, 13.6 without the dispatcher, 13.1 without working out the workspace's size a second
// time (see decode).
at::Tensor fresh(at::IntArrayRef sizes, const at::Tensor &like, at::ScalarType type)
{
    if (at::hasCallbacks())
        return at::empty(sizes, like.options().dtype(type));
    return at::cuda::empty(sizes, type, at::kStrided, like.device(), false, c10::nullopt);
}

PyObject *pair(at::Tensor &&a, at::Tensor &&b)
{
    PyObject *x = THPVariable_Wrap(std::move(a)), *y = THPVariable_Wrap(std::move(b));
    PyObject *r = x && y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    return r;
}

// rows read in place: channels contiguous, even strides, 4-byte aligned base
bool rows(const at::Tensor &t)
{
    const auto st = t.strides();
    for (size_t i = 0; i + 1 < st.size(); i++)
        if (st[i] % 2)
            return false;
    return st.back() == 1 && (uintptr_t)t.const_data_ptr() % 4 == 0;
}

// rope_qk(q, k, cos, sin)
PyObject *rope_qk(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 4 || !unwatched())
        Py_RETURN_NONE;
    const at::Tensor *t[4];
    for (int i = 0; i < 4; i++)
        if (!(t[i] = plain(args[i])) || t[i]->scalar_type() != t[0]->scalar_type() || t[i]->device() != t[0]->device())
            Py_RETURN_NONE;
    const at::Tensor &q = *t[0], &k = *t[1], &c = *t[2], &s = *t[3];
    if (!half_type(q) || q.dim() != 4 || k.dim() != 4 || c.dim() != 3 || s.dim() != 3)
        Py_RETURN_NONE;
    const int64_t B = q.size(0), Hq = q.size(1), T = q.size(2), D = q.size(3), H = k.size(1);
    if (k.size(0) != B || k.size(2) != T || k.size(3) != D || c.sizes() != s.sizes() || c.strides() != s.strides() ||
        c.size(1) != T || c.size(2) != D || (c.size(0) != 1 && c.size(0) != B) || D % 4 || B * Hq * T * D <= 0 || H <= 0 ||
        B * std::max(Hq, H) * T > INT32_MAX || !rows(q) || !rows(k) || !rows(c) || !rows(s))
        Py_RETURN_NONE;
    void *stream;
    if (!current(q.device(), stream))
        Py_RETURN_NONE;
    at::Tensor qo, ko;
    int rc;
    qo = fresh({B, Hq, T, D}, q, q.scalar_type());
    ko = fresh({B, H, T, D}, q, q.scalar_type());
    if (!qo.has_storage() || !ko.has_storage())
        Py_RETURN_NONE;
    void *qp = qo.mutable_data_ptr(), *kp = ko.mutable_data_ptr();
    Py_BEGIN_ALLOW_THREADS
    rc = adkv_rope_qk(q.const_data_ptr(), k.const_data_ptr(), c.const_data_ptr(), s.const_data_ptr(), qp, kp, (int)B, (int)Hq,
                      (int)H, (int)T, (int)D, q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
                      c.size(0) == B && B > 1 ? c.stride(0) : 0, c.stride(1), q.scalar_type() == at::kBFloat16, stream);
    Py_END_ALLOW_THREADS
    return rc ? PyLong_FromLong(rc) : pair(std::move(qo), std::move(ko));
}

// n contiguous tensors of `type` and `numel` elements each on `device` in a tuple -> their addresses
// (written: in place, so a storage shared by a lazy copy becomes the tensor's own)
bool pointers(PyObject *tuple, Py_ssize_t n, at::ScalarType type, int64_t numel, c10::Device device, const void **out,
              bool written = false)
{
    if (!PyTuple_CheckExact(tuple) || PyTuple_GET_SIZE(tuple) != n)
        return false;
    for (Py_ssize_t i = 0; i < n; i++) {
        const at::Tensor *p = plain(PyTuple_GET_ITEM(tuple, i));
        if (!p || p->scalar_type() != type || p->numel() != numel || !p->is_contiguous() || p->device() != device)
            return false;
        out[i] = written ? p->mutable_data_ptr() : p->const_data_ptr();
    }
    return true;
}

// both checkpoint tensors [B, H, n, D, 2] or neither
bool checkpoints(PyObject *const *args, int64_t B, int64_t H, int64_t D, long interval, long bits, c10::Device device, void **ck,
                 int64_t &n)
{
    ck[0] = ck[1] = nullptr;
    n = 0;
    if (args[0] == Py_None && args[1] == Py_None)
        return true;
    for (int i = 0; i < 2; i++) {
        const at::Tensor *c = plain(args[i]);
        if (!c || c->scalar_type() != at::kHalf || c->dim() != 5 || c->size(0) != B || c->size(1) != H || c->size(2) < 1 ||
            c->size(2) > INT32_MAX || c->size(3) != D || c->size(4) != 2 || !c->is_contiguous() || c->device() != device ||
            (i && c->size(2) != n) || interval <= 0 || interval % (32 / bits) || interval > INT32_MAX)
            return false;
        n = c->size(2);
        ck[i] = c->mutable_data_ptr();
    }
    return true;
}

// decode(q, k_new, v_new, params (ten), key codes, value codes, key checkpoints, value checkpoints, interval,
//        bits, T, scaling, mask or None, workspaces {(device index, stream): uint8 tensor})
PyObject *decode(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 14 || !unwatched() || !PyFloat_CheckExact(args[11]) ||
        !PyDict_CheckExact(args[13]))
        Py_RETURN_NONE;
    const at::Tensor *qt = plain(args[0]), *kn = plain(args[1]), *vn = plain(args[2]), *kc = plain(args[4]), *vc = plain(args[5]);
    if (!qt || !kn || !vn || !kc || !vc)
        Py_RETURN_NONE;
    const at::Tensor &q = *qt;
    const long interval = PyLong_AsLong(args[8]), bits = PyLong_AsLong(args[9]), T = PyLong_AsLong(args[10]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    if (!half_type(q) || kn->scalar_type() != q.scalar_type() || vn->scalar_type() != q.scalar_type() || q.dim() != 4 ||
        kc->dim() != 6 || kc->scalar_type() != at::kByte || vc->scalar_type() != at::kByte || kc->sizes() != vc->sizes() ||
        (bits != 2 && bits != 4) || T < 0 || T >= INT32_MAX)
        Py_RETURN_NONE;
    const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3), H = kc->size(1), n_super = kc->size(2);
    if (q.size(2) != 1 || B <= 0 || H <= 0 || kc->size(0) != B || kc->size(3) * 4 != D || kc->size(4) != 4 || kc->size(5) != 4 ||
        Hq % H || (Hq / H != 1 && Hq / H != 2 && Hq / H != 4 && Hq / H != 8) || (D != 128 && D != 256 && D != 512) ||
        ((Hq != H || bits != 4) && D != 128) || T / (32 / bits) >= n_super || n_super > INT32_MAX || B * Hq > INT32_MAX)
        Py_RETURN_NONE;
    const int64_t token[4] = {B, H, 1, D};
    if (kn->sizes() != at::IntArrayRef(token) || vn->sizes() != at::IntArrayRef(token) || !q.is_contiguous() || !kn->is_contiguous() || !vn->is_contiguous() ||
        !kc->is_contiguous() || !vc->is_contiguous())
        Py_RETURN_NONE;
    for (const at::Tensor *t : {kn, vn, kc, vc})
        if (t->device() != q.device())
            Py_RETURN_NONE;
    const void *params[10];
    void *ck[2];
    int64_t n_ckpt;
    if (!pointers(args[3], 10, at::kHalf, H * D, q.device(), params) ||
        !checkpoints(args + 6, B, H, D, interval, bits, q.device(), ck, n_ckpt))
        Py_RETURN_NONE;
    const int64_t n = T + 1;
    const at::Tensor *mask = nullptr;
    int rows_per_mask_row = 1, mask_type = -1; // the type as the kernels read it, -1: to fp32 first
    if (args[12] != Py_None) {
        mask = plain(args[12]);
        if (!mask || mask->device() != q.device() || !at::isFloatingType(mask->scalar_type()) ||
            (mask->dim() != 3 && !(mask->dim() == 4 && mask->size(2) == 1)) || mask->size(0) != B ||
            (mask->size(1) != 1 && mask->size(1) != Hq) || mask->size(-1) != n)
            Py_RETURN_NONE;
        rows_per_mask_row = mask->size(1) == 1 ? (int)Hq : 1;
        mask_type = mask->scalar_type() == at::kFloat ? ADKV_DT_F32 : mask->scalar_type() == at::kHalf ? ADKV_DT_F16
                    : mask->scalar_type() == at::kBFloat16 ? ADKV_DT_BF16 : -1;
    }
    void *stream;
    if (!current(q.device(), stream))
        Py_RETURN_NONE;
    PyObject *key = Py_BuildValue("(iN)", (int)q.device().index(), PyLong_FromVoidPtr(stream));
    PyObject *w = key ? PyDict_GetItem(args[13], key) : nullptr; // borrowed
    Py_XDECREF(key);
    const at::Tensor *ws = w ? plain(w) : nullptr;
    if (!ws || ws->scalar_type() != at::kByte || !ws->is_contiguous() || ws->device() != q.device())
        Py_RETURN_NONE;
    at::Tensor out, weights, m, scratch = *ws; // held: another thread may replace the dictionary's entry
    int rc;
    if (mask) {
        m = (mask_type >= 0 ? *mask : mask->to(at::kFloat)).contiguous();
        if (!m.has_storage())
            Py_RETURN_NONE;
    }
    const int64_t pitch = adkv_row_pitch((int)n);
    out = fresh({B, Hq, D}, q, q.scalar_type());
    weights = fresh({B, Hq, pitch}, q, at::kHalf);
    if (!out.has_storage() || !weights.has_storage())
        Py_RETURN_NONE;
    void *op = out.mutable_data_ptr(), *wp = weights.mutable_data_ptr(), *kcp = kc->mutable_data_ptr(), *vcp = vc->mutable_data_ptr(),
         *work = scratch.mutable_data_ptr(); // before the lock is given up: these may throw
    const void *mp = mask ? m.const_data_ptr() : nullptr;
    const double scaling = PyFloat_AS_DOUBLE(args[11]);
    Py_BEGIN_ALLOW_THREADS
    rc = adkv_decode_step(q.const_data_ptr(), kcp, vcp, kn->const_data_ptr(), vn->const_data_ptr(), params, params + 5, mp, rows_per_mask_row, (float)scaling, op, wp, pitch, (int)B,
                          (int)Hq, (int)H, (int)T, (int)D, (int)n_super, (int)bits,
                          (q.scalar_type() == at::kBFloat16 ? ADKV_DT_BF16 : ADKV_DT_F16) | ADKV_MASK_DT(std::max(mask_type, ADKV_DT_F32)),
                          ck[0], ck[1], (int)n_ckpt, (int)interval, work, scratch.numel(), stream);
    Py_END_ALLOW_THREADS
    if (rc == ADKV_E_WORKSPACE) // too small: said before anything is launched, and the Python function gets a larger one
        Py_RETURN_NONE;
    const int64_t sizes[3] = {B, Hq, n}, strides[3] = {Hq * pitch, pitch, 1};
    weights.unsafeGetTensorImpl()->set_sizes_and_strides(at::IntArrayRef(sizes), at::IntArrayRef(strides));
    return rc ? PyLong_FromLong(rc) : pair(std::move(out), std::move(weights));
}

// append(key codes, value codes, k rows, v rows, key params (five), value params (five), T0, key state,
//        value state, key checkpoints, value checkpoints, interval, bits, fresh)
PyObject *append(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 14 || !unwatched() || (args[13] != Py_True && args[13] != Py_False)) // any other truth value: Python's
        Py_RETURN_NONE;
    const at::Tensor *t[6];
    const int at_arg[6] = {0, 1, 2, 3, 7, 8};
    for (int i = 0; i < 6; i++)
        if (!(t[i] = plain(args[at_arg[i]])) || t[i]->device() != t[0]->device())
            Py_RETURN_NONE;
    const at::Tensor &kc = *t[0], &vc = *t[1], &k = *t[2], &v = *t[3];
    const long T0 = PyLong_AsLong(args[6]), interval = PyLong_AsLong(args[11]), bits = PyLong_AsLong(args[12]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const bool fresh = args[13] == Py_True;
    if (!half_type(k) || v.scalar_type() != k.scalar_type() || k.dim() != 4 || v.sizes() != k.sizes() || kc.dim() != 6 ||
        kc.scalar_type() != at::kByte || vc.scalar_type() != at::kByte || kc.sizes() != vc.sizes() || !kc.is_contiguous() ||
        !vc.is_contiguous() || (bits != 2 && bits != 4) || T0 < 0 || (fresh && T0 != 0))
        Py_RETURN_NONE;
    const int64_t B = k.size(0), H = k.size(1), n = k.size(2), D = k.size(3), n_super = kc.size(2), tps = 32 / bits;
    if (B <= 0 || H <= 0 || n <= 0 || kc.size(0) != B || kc.size(1) != H || kc.size(3) * 4 != D || kc.size(4) != 4 ||
        kc.size(5) != 4 || (D != 128 && D != 256 && D != 512) || (T0 + n + tps - 1) / tps > n_super || n_super * tps > INT32_MAX ||
        B * H > INT32_MAX / D)
        Py_RETURN_NONE;
    int64_t strides[2][3];
    for (int i = 0; i < 2; i++) {
        const at::Tensor &x = *t[2 + i];
        for (int j = 0; j < 3; j++)
            strides[i][j] = x.stride(j);
        if (!x.is_contiguous() && (!rows(x) || x.stride(2) < D || x.stride(0) < 0 || x.stride(1) < 0))
            Py_RETURN_NONE;
        const at::Tensor &st = *t[4 + i];
        if (st.scalar_type() != at::kHalf || !st.is_contiguous() || st.numel() != B * H * D * 2)
            Py_RETURN_NONE;
    }
    const void *kp[5], *vp[5];
    void *ck[2], *stream;
    int64_t n_ckpt;
    if (!pointers(args[4], 5, at::kHalf, H * D, kc.device(), kp) || !pointers(args[5], 5, at::kHalf, H * D, kc.device(), vp) ||
        !checkpoints(args + 9, B, H, D, interval, bits, kc.device(), ck, n_ckpt) || !current(kc.device(), stream))
        Py_RETURN_NONE;
    const int dtype = k.scalar_type() == at::kBFloat16 ? ADKV_DT_BF16 : ADKV_DT_F16;
    const int64_t *ks = k.is_contiguous() ? nullptr : strides[0], *vs = v.is_contiguous() ? nullptr : strides[1];
    const int iv = ck[0] ? (int)interval : 0;
    void *out[4] = {kc.mutable_data_ptr(), vc.mutable_data_ptr(), t[4]->mutable_data_ptr(), t[5]->mutable_data_ptr()};
    const void *in[2] = {k.const_data_ptr(), v.const_data_ptr()};
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fresh ? adkv_prefill_kv_pair(out[0], out[1], in[0], in[1], dtype, ks, vs, kp, vp, (int)B, (int)H, (int)n, (int)D,
                                      (int)n_super, (int)bits, out[2], out[3], ck[0], ck[1], (int)n_ckpt, iv, stream)
               : adkv_append_kv_pair(out[0], out[1], in[0], in[1], dtype, ks, vs, kp, vp, (int)B, (int)H, (int)T0, (int)n, (int)D,
                                     (int)n_super, (int)bits, out[2], out[3], ck[0], ck[1], (int)n_ckpt, iv, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// quant_f32(x, (alpha, beta, target, zp_init, sc_init), lower, upper, sc_min, sc_max, output_states, free_params)
//   -> (xhat, zp sequence or None, sc sequence or None)
PyObject *quant_f32(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 8 || !unwatched() || !PyFloat_CheckExact(args[4]) || !PyFloat_CheckExact(args[5]))
        Py_RETURN_NONE;
    const at::Tensor *x = plain(args[0]);
    const long lower = PyLong_AsLong(args[2]), upper = PyLong_AsLong(args[3]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    if (!x || x->dim() != 3 || !x->is_contiguous() || (!half_type(*x) && x->scalar_type() != at::kFloat))
        Py_RETURN_NONE;
    const int64_t B = x->size(0), T = x->size(1), C = x->size(2);
    const void *p[5];
    void *stream;
    if (B <= 0 || T <= 0 || C <= 0 || B > INT32_MAX || T > INT32_MAX || C > INT32_MAX || lower < INT32_MIN || upper > INT32_MAX ||
        !pointers(args[1], 5, at::kFloat, C, x->device(), p) || !current(x->device(), stream))
        Py_RETURN_NONE;
    at::Tensor out, state, seq[2];
    int rc;
    out = fresh({B, T, C}, *x, x->scalar_type());
    state = fresh({2, B, C}, *x, at::kFloat);
    if (args[6] == Py_True)
        for (at::Tensor &t : seq)
            t = fresh({B, T, C}, *x, at::kFloat);
    if (!out.has_storage() || !state.has_storage())
        Py_RETURN_NONE;
    void *op = out.mutable_data_ptr(), *zp = state.mutable_data_ptr(), *sc = (float *)zp + B * C;
    void *sp[2] = {seq[0].defined() ? seq[0].mutable_data_ptr() : nullptr, seq[1].defined() ? seq[1].mutable_data_ptr() : nullptr};
    const int type = (x->scalar_type() == at::kFloat ? ADKV_DT_F32 : x->scalar_type() == at::kHalf ? ADKV_DT_F16 : ADKV_DT_BF16) |
                     (args[7] == Py_True ? ADKV_PARAMS_FREE : 0);
    const double lo = PyFloat_AS_DOUBLE(args[4]), hi = PyFloat_AS_DOUBLE(args[5]);
    Py_BEGIN_ALLOW_THREADS
    rc = adkv_quant_f32(x->const_data_ptr(), op, nullptr, zp, sc, p[3], p[4], p[0], p[1], p[2], sp[0], sp[1], (int)B, (int)T, (int)C,
                        T * C, C, type, (int)lower, (int)upper, (float)lo, (float)hi, stream);
    Py_END_ALLOW_THREADS
    if (rc)
        return PyLong_FromLong(rc);
    PyObject *o = THPVariable_Wrap(std::move(out));
    PyObject *z = seq[0].defined() ? THPVariable_Wrap(std::move(seq[0])) : (Py_INCREF(Py_None), Py_None);
    PyObject *c = seq[1].defined() ? THPVariable_Wrap(std::move(seq[1])) : (Py_INCREF(Py_None), Py_None);
    PyObject *r = o && z && c ? PyTuple_Pack(3, o, z, c) : nullptr;
    Py_XDECREF(o);
    Py_XDECREF(z);
    Py_XDECREF(c);
    return r;
}

// quant_f32_pair(k rows, v rows, k out, v out, params (six), states (four), initial states (four) or None, lower,
//                upper, sc_min, sc_max)
PyObject *quant_f32_pair(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 11 || !unwatched() || !PyFloat_CheckExact(args[9]) || !PyFloat_CheckExact(args[10]))
        Py_RETURN_NONE;
    const at::Tensor *t[4];
    for (int i = 0; i < 4; i++)
        if (!(t[i] = plain(args[i])) || t[i]->dim() != 3 || t[i]->sizes() != t[0]->sizes() ||
            t[i]->scalar_type() != t[0]->scalar_type() || t[i]->stride(2) != 1 || t[i]->device() != t[0]->device())
            Py_RETURN_NONE;
    const at::Tensor &x = *t[0];
    const long lower = PyLong_AsLong(args[7]), upper = PyLong_AsLong(args[8]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const int64_t B = x.size(0), T = x.size(1), C = x.size(2);
    if ((!half_type(x) && x.scalar_type() != at::kFloat) || B <= 0 || T <= 0 || C <= 0 || B > INT32_MAX || T > INT32_MAX ||
        C > INT32_MAX || lower < INT32_MIN || upper > INT32_MAX)
        Py_RETURN_NONE;
    const void *rows[4], *params[6], *state[4], *init[4];
    int64_t strides[8];
    for (int i = 3; i >= 0; i--) { // outputs first (they may be the inputs); of a single sequence or token the strides may be anything
        rows[i] = i >= 2 ? t[i]->mutable_data_ptr() : t[i]->const_data_ptr();
        strides[2 * i] = B > 1 ? t[i]->stride(0) : T * std::max(t[i]->stride(1), C);
        strides[2 * i + 1] = T > 1 ? t[i]->stride(1) : C;
    }
    void *stream;
    for (Py_ssize_t i = 0; PyTuple_CheckExact(args[5]) && i < PyTuple_GET_SIZE(args[5]); i++) {
        const at::Tensor *st = plain(PyTuple_GET_ITEM(args[5], i));
        if (!st || st->dim() != 2 || st->size(0) != B)
            Py_RETURN_NONE;
    }
    if (!pointers(args[4], 6, at::kFloat, C, x.device(), params) || !pointers(args[5], 4, at::kFloat, B * C, x.device(), state, true) ||
        (args[6] != Py_None && !pointers(args[6], 4, at::kFloat, C, x.device(), init)) || !current(x.device(), stream))
        Py_RETURN_NONE;
    const int type = x.scalar_type() == at::kFloat ? ADKV_DT_F32 : x.scalar_type() == at::kHalf ? ADKV_DT_F16 : ADKV_DT_BF16;
    const double lo = PyFloat_AS_DOUBLE(args[9]), hi = PyFloat_AS_DOUBLE(args[10]);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = adkv_quant_f32_pair(rows, strides, const_cast<void *const *>(rows + 2), strides + 4, const_cast<void *const *>(state),
                             args[6] != Py_None ? init : nullptr, params, (int)B, (int)T, (int)C, type, (int)lower, (int)upper,
                             (float)lo, (float)hi, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// No C++ exception reaches Python's frames.
template <PyObject *(*CALL)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *self, PyObject *const *args, Py_ssize_t n)
{
    try {
        return CALL(self, args, n);
    } catch (const std::exception &) {
        Py_RETURN_NONE; // out of memory, or a mode that allocates otherwise: the Python function meets it too
    }
}

PyObject *init(PyObject *, PyObject *f)
{
    Py_INCREF(f);
    Py_XSETREF(raw_stream, f);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"init", init, METH_O, "init(function from device index to raw stream)"},
    {"rope_qk", (PyCFunction)(void (*)(void))guarded<rope_qk>, METH_FASTCALL, nullptr},
    {"decode", (PyCFunction)(void (*)(void))guarded<decode>, METH_FASTCALL, nullptr},
    {"append", (PyCFunction)(void (*)(void))guarded<append>, METH_FASTCALL, nullptr},
    {"quant_f32", (PyCFunction)(void (*)(void))guarded<quant_f32>, METH_FASTCALL, nullptr},
    {"quant_f32_pair", (PyCFunction)(void (*)(void))guarded<quant_f32_pair>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }

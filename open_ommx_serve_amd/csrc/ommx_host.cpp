// Native half of the Python launchers: argument checks, workspace and kernel launches of one call
// in one C++ function, so that a call costs a few microseconds of host time instead of tens (a
// decode step of a short context is 13 us of GPU time; checking its ~40 arguments tensor by tensor in
// Python took 33 us).
//
// Contract with the Python side: a function here returns True when it has launched the call and
// False when anything about the arguments is not exactly what it expects; it then has launched and
// changed nothing, and the Python caller goes through its own checks, which raise the exception that
// names the problem or bring the arguments into the expected form.  A failing launch raises
// RuntimeError.  Every check that the Python side makes is made here too.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/Allocator.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <atomic>

#include "../../include/ommx_hip.h"

namespace {

// ── argument readers: every one reports a mismatch through `ok` ────────────────────────────────

const at::Tensor* as_tensor(PyObject* o, bool& ok) {
    if (!THPVariable_Check(o)) { ok = false; return nullptr; }
    return &THPVariable_Unpack(o);
}
const at::Tensor* as_tensor_or_none(PyObject* o, bool& ok) { return o == Py_None ? nullptr : as_tensor(o, ok); }

int64_t as_int(PyObject* o, bool& ok) {
    if (!PyLong_Check(o)) { ok = false; return 0; }
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow || v > INT32_MAX || v < INT32_MIN) ok = false;      // the C ABI takes int
    return v;
}
double as_double(PyObject* o, bool& ok) {
    if (PyFloat_Check(o)) return PyFloat_AS_DOUBLE(o);
    return static_cast<double>(as_int(o, ok));
}
bool as_bool(PyObject* o, bool& ok) {
    if (o != Py_True && o != Py_False) ok = false;
    return o == Py_True;
}
bool is_word(PyObject* o, const char* w) { return PyUnicode_Check(o) && PyUnicode_CompareWithASCIIString(o, w) == 0; }

bool is_group_size(int64_t g) { return g == 16 || g == 32 || g == 64 || g == 128; }
template <class T = void>
T* data(const at::Tensor* t) { return t ? static_cast<T*>(t->data_ptr()) : nullptr; }

bool failed(int rc, const char* what) {
    if (rc == 0) return false;
    PyErr_Format(PyExc_RuntimeError, "%s failed (rc=%d): %s", what, rc, ommx_last_error());
    return true;
}

int cu_count(int device) {
    static std::atomic<int> known[64];
    if (device < 0 || device >= 64) return 256;
    int n = known[device].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) n = 256;
        known[device].store(n, std::memory_order_relaxed);
    }
    return n;
}

// ── split count ────────────────────────────────────────────────────────────────────────────────

// The rule that paged_decode.auto_num_kv_splits documents.
int auto_splits(int64_t max_seq, int64_t batch, int64_t kv_heads, int64_t n_cu, int64_t group_tokens,
                double mean_seq /* < 0: not given */, int resident) {
    constexpr int64_t kMax = 512;
    const int64_t wgs = std::max<int64_t>(1, batch * std::max<int64_t>(1, kv_heads / 4));
    const int64_t gt = std::max<int64_t>(32, group_tokens), step = std::max<int64_t>(64, gt);
    const int64_t steps = std::max<int64_t>(1, (max_seq + step - 1) / step);
    const int64_t groups = std::max<int64_t>(1, (max_seq + gt - 1) / gt);
    const bool equal = batch == 1 || (mean_seq >= 0 && mean_seq >= 0.9 * static_cast<double>(max_seq));
    auto count = [&](int64_t res) {
        int64_t want = std::max<int64_t>(1, std::min(kMax, ((equal ? 1 : 2) * res * n_cu) / wgs));
        if (!equal && batch > 1) {
            const int64_t n = std::min(want, steps);
            if ((steps + n - 1) / n > 16) want = std::max<int64_t>(1, std::min(kMax, (4 * res * n_cu) / wgs));
        }
        return want;
    };
    int64_t res = std::max(1, resident), want = count(res);
    if (res >= 3 && steps < 4 * want) { res = 2; want = count(res); }
    if (want >= 2 * steps) return static_cast<int>(std::min(want, groups));
    if (res >= 3) return static_cast<int>(std::max<int64_t>(1, std::min(want, groups)));
    const int64_t target = std::max<int64_t>(1, std::min(want, steps));
    const int64_t per = (steps + target - 1) / target;
    return static_cast<int>((steps + per - 1) / per);
}

PyObject* py_auto_splits(PyObject*, PyObject* const* a, Py_ssize_t n) {
    bool ok = n == 7;
    if (!ok) { PyErr_SetString(PyExc_TypeError, "auto_num_kv_splits takes 7 arguments"); return nullptr; }
    const int64_t max_seq = as_int(a[0], ok), batch = as_int(a[1], ok), heads = as_int(a[2], ok),
                  n_cu = as_int(a[3], ok), gt = as_int(a[4], ok);
    const double mean = as_double(a[5], ok);
    const int64_t res = as_int(a[6], ok);
    if (!ok) { PyErr_SetString(PyExc_ValueError, "auto_num_kv_splits: integers expected"); return nullptr; }
    return PyLong_FromLong(auto_splits(max_seq, batch, heads, n_cu, gt, mean, static_cast<int>(res)));
}

// ── decode ─────────────────────────────────────────────────────────────────────────────────────

enum DecodeArg {
    A_Q, A_KBASE, A_KSCALE, A_KZP, A_KOIDX, A_KOVAL, A_VMAIN, A_VSCALE, A_VZP, A_KTAIL, A_VTAIL, A_BTAIL,
    A_O, A_LSE, A_RT, A_RG, A_SEQ,
    A_SM, A_PS, A_CAP, A_KOUT, A_KFMT, A_COMBI, A_BITMAP, A_KOBMP, A_MS, A_MC, A_MAP, A_INT8, A_SPLITS,
    A_MAXSEQ, A_MAXTAIL, A_WS, A_OFF, A_GBASE, A_FORCE, A_MEAN, A_ERR, A_COUNT
};

bool is_shape3(const at::Tensor& t, int64_t a, int64_t b, int64_t c) {
    return t.dim() == 3 && t.size(0) == a && t.size(1) == b && t.size(2) == c;
}
bool on(const at::Tensor* t, c10::Device d) { return t && t->device() == d; }

PyObject* py_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != A_COUNT) { PyErr_SetString(PyExc_TypeError, "decode: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *q = as_tensor(a[A_Q], ok), *k_base = as_tensor(a[A_KBASE], ok),
                     *k_scale = as_tensor(a[A_KSCALE], ok), *k_zp = as_tensor(a[A_KZP], ok),
                     *k_oidx = as_tensor_or_none(a[A_KOIDX], ok), *k_oval = as_tensor_or_none(a[A_KOVAL], ok),
                     *v_main = as_tensor(a[A_VMAIN], ok), *v_scale = as_tensor(a[A_VSCALE], ok),
                     *v_zp = as_tensor(a[A_VZP], ok), *k_tail = as_tensor_or_none(a[A_KTAIL], ok),
                     *v_tail = as_tensor_or_none(a[A_VTAIL], ok), *b_tail = as_tensor_or_none(a[A_BTAIL], ok),
                     *o = as_tensor(a[A_O], ok), *lse = as_tensor(a[A_LSE], ok), *rt = as_tensor(a[A_RT], ok),
                     *rg = as_tensor(a[A_RG], ok), *seq = as_tensor(a[A_SEQ], ok),
                     *k_obmp = as_tensor_or_none(a[A_KOBMP], ok), *ms = as_tensor_or_none(a[A_MS], ok),
                     *mc = as_tensor_or_none(a[A_MC], ok), *ws = as_tensor_or_none(a[A_WS], ok),
                     *err = as_tensor_or_none(a[A_ERR], ok);
    const double sm_scale = as_double(a[A_SM], ok), cap = as_double(a[A_CAP], ok);
    const int64_t ps = as_int(a[A_PS], ok), k = as_int(a[A_KOUT], ok), off = as_int(a[A_OFF], ok),
                  gbase = as_int(a[A_GBASE], ok);
    const bool bitmap = as_bool(a[A_BITMAP], ok), int8 = as_bool(a[A_INT8], ok), force = as_bool(a[A_FORCE], ok);
    const bool combinadic = as_bool(a[A_COMBI], ok), want_map = as_bool(a[A_MAP], ok);
    const int64_t given_splits = a[A_SPLITS] == Py_None ? 0 : as_int(a[A_SPLITS], ok);
    const int64_t max_seq = a[A_MAXSEQ] == Py_None ? -1 : std::max<int64_t>(1, as_int(a[A_MAXSEQ], ok));
    const int64_t max_tail = a[A_MAXTAIL] == Py_None ? 1 : as_int(a[A_MAXTAIL], ok);
    const double mean = a[A_MEAN] == Py_None ? -1.0 : as_double(a[A_MEAN], ok);
    ok = ok && !combinadic && (is_word(a[A_KFMT], "i2f4") || is_word(a[A_KFMT], "itf4"));
    if (!ok) Py_RETURN_FALSE;

    // geometry of the planes
    if (q->dim() != 3 || k_base->dim() != 4 || k_scale->dim() != 3 || v_main->dim() != 4 || v_scale->dim() != 4 ||
        v_zp->dim() != 4 || ps < 1)
        Py_RETURN_FALSE;
    const c10::Device dev = q->device();
    if (!dev.is_cuda()) Py_RETURN_FALSE;
    const int64_t pages = k_base->size(0), slots = k_scale->size(0), B = q->size(0), Hq = q->size(1),
                  Hkv = k_base->size(2), D = k_base->size(3) * 4;
    const int64_t gt = (pages == 0 || slots == 0) ? 32 : pages * ps / slots;
    const bool v_bf16 = v_main->scalar_type() == at::kBFloat16;
    const int64_t v_width = v_bf16 ? v_main->size(3) : v_main->size(3) * 4, per_row = v_scale->size(3);
    const int64_t gc = per_row == 0 ? 32 : v_width / per_row;
    if (!is_group_size(gt) || !is_group_size(gc) || v_width % gc || B < 1 || Hkv < 1 || Hq < Hkv || Hq % Hkv ||
        v_width != D || (D != 64 && D != 128) || q->size(2) != D || gt % ps || pages > INT32_MAX || slots > INT32_MAX)
        Py_RETURN_FALSE;
    const int64_t R = Hq / Hkv;
    if (R != 1 && R != 2 && R != 4 && R != 8) Py_RETURN_FALSE;
    for (const at::Tensor* t : {k_base, v_main, v_scale, v_zp})
        if (!t->is_contiguous() || t->size(0) != pages || t->size(1) != ps || t->size(2) != Hkv) Py_RETURN_FALSE;
    if (!is_shape3(*k_scale, slots, Hkv, D) || !is_shape3(*k_zp, slots, Hkv, D) ||
        k_zp->scalar_type() != at::kBFloat16 || !is_shape3(*o, B, Hq, D) || lse->dim() != 2 || lse->size(0) != B ||
        lse->size(1) != Hq)
        Py_RETURN_FALSE;
    const at::ScalarType st = k_scale->scalar_type();
    const bool scale_bf16 = st == at::kBFloat16;
    if (st != v_scale->scalar_type() || (st != at::kChar && !scale_bf16) || scale_bf16 == int8) Py_RETURN_FALSE;
    if (q->scalar_type() != at::kBFloat16 || q->stride(2) != 1) Py_RETURN_FALSE;

    // lengths, tables, outputs
    if (seq->numel() < B || !seq->is_contiguous() || seq->scalar_type() != at::kInt) Py_RETURN_FALSE;
    if (b_tail && (b_tail->numel() < B || !b_tail->is_contiguous() || b_tail->scalar_type() != at::kInt)) Py_RETURN_FALSE;
    if (rt->dim() != 2 || rg->dim() != 2 || rt->size(0) < B || rg->size(0) < B ||
        rt->scalar_type() != rg->scalar_type() || (rt->scalar_type() != at::kInt && rt->scalar_type() != at::kLong) ||
        rt->stride(1) != 1 || rg->stride(1) != 1)
        Py_RETURN_FALSE;
    if (o->scalar_type() != at::kFloat || lse->scalar_type() != at::kFloat || o->stride(2) != 1 || lse->stride(1) != 1)
        Py_RETURN_FALSE;
    for (const at::Tensor* t : {k_base, k_scale, v_main, o, lse, rt, rg, seq})
        if (!on(t, dev)) Py_RETURN_FALSE;
    if (off < 0 || off >= ps || gbase < 0) Py_RETURN_FALSE;

    // outliers
    const at::Tensor* k_index = bitmap ? k_obmp : k_oidx;
    const bool own_map = want_map && k > 0;
    if (k < 0 || k > 16 || (bitmap && k > 8)) Py_RETURN_FALSE;
    if (k > 0) {
        const int64_t index_bytes = bitmap ? (gt + 7) / 8 : (7 * k + 7) / 8;
        for (const at::Tensor* t : {k_oval, k_index})
            if (!t || t->scalar_type() != at::kByte || t->dim() != 4 || t->size(0) != slots || t->size(1) != Hkv ||
                t->size(2) != D || t->size(3) != (t == k_oval ? (k + 1) / 2 : index_bytes) || !t->is_contiguous())
                Py_RETURN_FALSE;
    }
    if (own_map && (!ms || !mc)) Py_RETURN_FALSE;
    for (const at::Tensor* t : {ms, mc})
        if (t && (!t->is_contiguous() ||
                  (own_map && (t->scalar_type() != at::kBFloat16 || !is_shape3(*t, slots, Hkv, D)))))
            Py_RETURN_FALSE;
    if (!k_scale->is_contiguous() || !k_zp->is_contiguous()) Py_RETURN_FALSE;

    // tail
    const bool tail = gbase == 0 && k_tail && v_tail && b_tail && k_tail->dim() == 4 && k_tail->size(1) > 0 && max_tail > 0;
    if (gbase == 0 && k_tail && v_tail && b_tail && k_tail->dim() != 4) Py_RETURN_FALSE;
    if (tail && (k_tail->scalar_type() != at::kBFloat16 || v_tail->scalar_type() != at::kBFloat16 ||
                 k_tail->stride(3) != 1 || v_tail->dim() != 4 || v_tail->stride(3) != 1 ||
                 k_tail->sizes() != v_tail->sizes() || k_tail->size(0) < B || k_tail->size(2) != Hkv ||
                 k_tail->size(3) != D))
        Py_RETURN_FALSE;
    if (err && (err->scalar_type() != at::kInt || !on(err, dev))) Py_RETURN_FALSE;

    // splits and the workspace of their partial states
    if (given_splits < 0 || (a[A_SPLITS] == Py_None && max_seq < 0)) Py_RETURN_FALSE;
    int64_t S = std::max<int64_t>(1, given_splits);
    if (a[A_SPLITS] == Py_None) {
        // The serving-recipe kernel keeps three workgroups per compute unit resident with up to 4 q heads per
        // kv head (two with 8, and so do the other kernels); at head_dim 64 one of its waves takes a pair of kv heads.
        const bool plain_planes = gt == 32 && gc == 32 && !scale_bf16 && !v_bf16 && !force;
        const bool lean = plain_planes && ((D == 128 && R <= 4 && k == 6) ||
                                           (bitmap && k >= 1 && k <= 6 && ((D == 128 && R <= 4) ||
                                                                           (D == 64 && R <= 2 && Hkv % 2 == 0))));
        const bool paired = plain_planes && D == 64 && bitmap && k >= 1 && k <= 8 && R <= 4 && Hkv % 2 == 0;
        S = auto_splits(max_seq, B, paired ? Hkv / 2 : Hkv, cu_count(dev.index()), gt, mean, lean ? 3 : 2);
    }
    if (ws && (ws->scalar_type() != at::kFloat || ws->dim() != 4 || ws->size(0) != B || ws->size(1) != Hq ||
               ws->size(2) < S || ws->size(3) < D + 1 || ws->stride(3) != 1))
        Py_RETURN_FALSE;

    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
    int64_t al_b = Hq * (S + 1) * (D + 1), al_h = (S + 1) * (D + 1), al_s = D + 1;
    c10::DataPtr scratch;
    float* al;
    if (ws) {
        al = ws->data_ptr<float>();
        al_b = ws->stride(0); al_h = ws->stride(1); al_s = ws->stride(2);
    } else {
        scratch = c10::GetAllocator(c10::DeviceType::CUDA)->allocate(static_cast<size_t>(B * al_b) * sizeof(float));
        al = static_cast<float*>(scratch.get());
    }
    const uint16_t* qp = data<const uint16_t>(q);
    int rc, rc2 = 0;
    Py_BEGIN_ALLOW_THREADS
    rc = (force ? ommx_decode_splitkv_ref : ommx_decode_splitkv)(
        qp, q->stride(0), q->stride(1), data<uint8_t>(k_base), data(k_scale), data<uint16_t>(k_zp),
        own_map ? data<uint16_t>(ms) : nullptr, own_map ? data<uint16_t>(mc) : nullptr,
        k > 0 ? data<uint8_t>(k_index) : nullptr, k > 0 ? data<uint8_t>(k_oval) : nullptr, data<uint8_t>(v_main),
        data(v_scale), data<uint16_t>(v_zp), data(rt), rt->stride(0), data(rg), rg->stride(0),
        rt->scalar_type() == at::kLong, data<int32_t>(seq), al, al_b, al_h, al_s, B, Hq, Hkv, D, ps, k,
        bitmap ? OMMX_INDEX_BITMAP : OMMX_INDEX_RELIDX7, scale_bf16, gt, gc, v_bf16, S, sm_scale, cap, off, gbase,
        pages, slots, data<int32_t>(err), stream);
    if (rc == 0)
        rc2 = ommx_decode_combine(
            al, al_b, al_h, al_s, qp, q->stride(0), q->stride(1), tail ? data<uint16_t>(k_tail) : nullptr,
            tail ? data<uint16_t>(v_tail) : nullptr, tail ? k_tail->stride(0) : 0, tail ? k_tail->stride(1) : 0,
            tail ? k_tail->stride(2) : 0, tail ? v_tail->stride(0) : 0, tail ? v_tail->stride(1) : 0,
            tail ? v_tail->stride(2) : 0, tail ? data<int32_t>(b_tail) : nullptr, data<int32_t>(seq),
            data<float>(o), o->stride(0), o->stride(1), data<float>(lse), lse->stride(0), B, Hq, Hkv, D, S, gt,
            tail ? k_tail->size(1) : 0, sm_scale, cap, stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "ommx_decode_splitkv") || failed(rc2, "ommx_decode_combine")) return nullptr;
    Py_RETURN_TRUE;
}

PyMethodDef methods[] = {
    {"auto_num_kv_splits", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_auto_splits)), METH_FASTCALL, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_decode)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ommx_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ommx_host(void) { return PyModule_Create(&module); }

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
#include <ATen/EmptyTensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/CachingHostAllocator.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/Allocator.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <initializer_list>
#include <mutex>
#include <random>
#include <vector>

#include "../../include/ommx_hip.h"
#include "ommx_internal.h"

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

// Whether nobody but the caller has a part in a call on these tensors.  A tracer, a transform (vmap, grad, forward
// mode, functionalisation), a dispatch or function mode, a tensor subclass and autograd all work in torch's
// dispatcher, which a launcher here goes past: they would miss its result or take it for a constant.  So what the
// dispatcher would look at for this call is held against the keys of an ordinary one.
bool plain_call(PyObject* const* a, Py_ssize_t n) {
    using c10::DispatchKey;
    static const c10::DispatchKeySet ordinary{
        DispatchKey::CPU, DispatchKey::CUDA, DispatchKey::AutogradCPU, DispatchKey::AutogradCUDA,
        DispatchKey::ADInplaceOrView, DispatchKey::BackendSelect, DispatchKey::AutocastCPU, DispatchKey::AutocastCUDA};
    if (at::impl::torch_function_mode_enabled()) return false;
    const c10::impl::LocalDispatchKeySet tls = c10::impl::tls_local_dispatch_key_set();
    const bool grad = c10::GradMode::is_enabled();
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (a[i] == Py_None) continue;
        if (!THPVariable_CheckExact(a[i])) return false;
        const at::Tensor& t = THPVariable_Unpack(a[i]);
        if (!ordinary.isSupersetOf((t.key_set() | tls.included_) - tls.excluded_) || (grad && t.requires_grad()) ||
            t._fw_grad(0).defined())
            return false;
    }
    return true;
}

// A tensor that a launch has written: autograd has to know that what it saved of it is gone.
void written(const at::Tensor& t) {
    if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
}

// The memory that a tensor spans (strides are never negative), empty without elements.
struct Span {
    const char *begin = nullptr, *end = nullptr;
    explicit Span(const at::Tensor& t) {
        if (t.numel() == 0) return;
        int64_t last = 0;
        for (int64_t d = 0; d < t.dim(); ++d) last += (t.size(d) - 1) * t.stride(d);
        begin = static_cast<const char*>(t.data_ptr());
        end = begin + (last + 1) * static_cast<int64_t>(t.element_size());
    }
    bool meets(const Span& o) const { return begin < o.end && o.begin < end; }
};
// Whether the memory that two tensors span has bytes in common.
bool share_memory(const at::Tensor& a, const at::Tensor& b) { return Span(a).meets(Span(b)); }

bool failed(int rc, const char* what) {
    if (rc == 0) return false;
    PyErr_Format(PyExc_RuntimeError, "%s failed (rc=%d): %s", what, rc, ommx_last_error());
    return true;
}

hipStream_t stream_of(c10::Device dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

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

PyObject* py_auto_num_kv_splits(PyObject*, PyObject* const* a, Py_ssize_t n) {
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

// One decode call: what both Python entries below fill in.
struct DecodeCall {
    const at::Tensor *q = nullptr, *k_base = nullptr, *k_scale = nullptr, *k_zp = nullptr, *k_index = nullptr,
                     *k_oval = nullptr, *v_main = nullptr, *v_scale = nullptr, *v_zp = nullptr, *k_tail = nullptr,
                     *v_tail = nullptr, *b_tail = nullptr, *o = nullptr, *lse = nullptr, *rt = nullptr, *rg = nullptr,
                     *seq = nullptr, *ms = nullptr, *mc = nullptr, *ws = nullptr, *err = nullptr;
    double sm_scale = 1, cap = 0, mean = -1;             // mean < 0: not given
    int64_t ps = 16, k = 0, splits = 0, max_seq = -1, max_tail = 1, off = 0, gbase = 0;   // splits 0 / max_seq < 0: not given
    bool bitmap = false, want_map = false, int8 = false, force = false;
    // tail rows read in place from the row history (k_tail / v_tail are [requests, rows, Hkv, D] then)
    const at::Tensor *hist_seq = nullptr, *hist_slots = nullptr;
    int64_t ring_sink = 0, ring_span = 0, win_sink = 0, win_recent = 0;
};

// Whether the history's ring holds every row that the window can ask for (what the merge over a history checks too).
bool hist_window_fits(const DecodeCall& c, int64_t gt, int64_t rows) {
    const int64_t most = c.win_recent + gt - 1;
    return c.win_sink >= 0 && c.win_recent >= 0 && rows > 0 &&
           (c.ring_span <= 0 ||
            (c.ring_sink == c.win_sink && c.ring_span >= most && c.ring_sink + c.ring_span <= rows));
}

// Checks the call and launches it: 1 launched, 0 refused (nothing done), -1 a launch failed (exception set).
int run_decode(const DecodeCall& c) {
    const at::Tensor &q = *c.q, &k_base = *c.k_base, &k_scale = *c.k_scale, &v_main = *c.v_main, &v_scale = *c.v_scale;
    // geometry of the planes
    if (q.dim() != 3 || k_base.dim() != 4 || k_scale.dim() != 3 || v_main.dim() != 4 || v_scale.dim() != 4 ||
        c.v_zp->dim() != 4 || c.ps < 1)
        return 0;
    const c10::Device dev = q.device();
    if (!dev.is_cuda()) return 0;
    const int64_t ps = c.ps, k = c.k, pages = k_base.size(0), slots = k_scale.size(0), B = q.size(0), Hq = q.size(1),
                  Hkv = k_base.size(2), D = k_base.size(3) * 4;
    const int64_t gt = (pages == 0 || slots == 0) ? 32 : pages * ps / slots;
    const bool v_bf16 = v_main.scalar_type() == at::kBFloat16;
    const int64_t v_width = v_bf16 ? v_main.size(3) : v_main.size(3) * 4, per_row = v_scale.size(3);
    const int64_t gc = per_row == 0 ? 32 : v_width / per_row;
    if (!is_group_size(gt) || !is_group_size(gc) || v_width % gc || B < 1 || Hkv < 1 || Hq < Hkv || Hq % Hkv ||
        v_width != D || (D != 64 && D != 128) || q.size(2) != D || gt % ps || pages > INT32_MAX || slots > INT32_MAX)
        return 0;
    const int64_t R = Hq / Hkv;
    if (R != 1 && R != 2 && R != 4 && R != 8) return 0;
    for (const at::Tensor* t : {c.k_base, c.v_main, c.v_scale, c.v_zp})
        if (!t->is_contiguous() || t->size(0) != pages || t->size(1) != ps || t->size(2) != Hkv) return 0;
    if (!is_shape3(k_scale, slots, Hkv, D) || !is_shape3(*c.k_zp, slots, Hkv, D) ||
        c.k_zp->scalar_type() != at::kBFloat16 || !is_shape3(*c.o, B, Hq, D))
        return 0;
    const at::ScalarType st = k_scale.scalar_type();
    const bool scale_bf16 = st == at::kBFloat16;
    if (st != v_scale.scalar_type() || (st != at::kChar && !scale_bf16) || scale_bf16 == c.int8) return 0;
    if (q.scalar_type() != at::kBFloat16 || q.stride(2) != 1) return 0;

    // (the workgroups of the merge that writes a row's halves both read all of it)
    if (c.hist_seq && share_memory(*c.o, q)) return 0;

    // lengths, tables, outputs
    if (c.seq->numel() < B || !c.seq->is_contiguous() || c.seq->scalar_type() != at::kInt) return 0;
    if (c.b_tail && (c.b_tail->numel() < B || !c.b_tail->is_contiguous() || c.b_tail->scalar_type() != at::kInt)) return 0;
    const at::Tensor &rt = *c.rt, &rg = *c.rg;
    if (rt.dim() != 2 || rg.dim() != 2 || rt.size(0) < B || rg.size(0) < B || rt.scalar_type() != rg.scalar_type() ||
        (rt.scalar_type() != at::kInt && rt.scalar_type() != at::kLong) || rt.stride(1) != 1 || rg.stride(1) != 1)
        return 0;
    const bool hist = c.hist_seq != nullptr;
    const bool o_bf16 = c.o->scalar_type() == at::kBFloat16;
    if ((c.o->scalar_type() != at::kFloat && !(hist && o_bf16)) || c.o->stride(2) != 1) return 0;
    if (!c.lse && !hist) return 0;
    if (c.lse && (c.lse->dim() != 2 || c.lse->size(0) != B || c.lse->size(1) != Hq ||
                  c.lse->scalar_type() != at::kFloat || c.lse->stride(1) != 1 || !on(c.lse, dev)))
        return 0;
    for (const at::Tensor* t : {c.k_base, c.k_scale, c.v_main, c.o, c.rt, c.rg, c.seq})
        if (!on(t, dev)) return 0;
    if (c.off < 0 || c.off >= ps || c.gbase < 0) return 0;

    // outliers
    const bool own_map = c.want_map && k > 0;
    if (k < 0 || k > 16 || (c.bitmap && k > 8)) return 0;
    if (k > 0) {
        const int64_t index_bytes = c.bitmap ? (gt + 7) / 8 : (7 * k + 7) / 8;
        for (const at::Tensor* t : {c.k_oval, c.k_index})
            if (!t || t->scalar_type() != at::kByte || t->dim() != 4 || t->size(0) != slots || t->size(1) != Hkv ||
                t->size(2) != D || t->size(3) != (t == c.k_oval ? (k + 1) / 2 : index_bytes) || !t->is_contiguous())
                return 0;
    }
    if (own_map && (!c.ms || !c.mc)) return 0;
    for (const at::Tensor* t : {c.ms, c.mc})
        if (t && (!t->is_contiguous() ||
                  (own_map && (t->scalar_type() != at::kBFloat16 || !is_shape3(*t, slots, Hkv, D)))))
            return 0;
    if (!k_scale.is_contiguous() || !c.k_zp->is_contiguous()) return 0;

    // tail
    const at::Tensor *kt = c.k_tail, *vt = c.v_tail;
    bool tail = false;
    if (hist) {
        if (!kt || !vt || kt->dim() != 4 || kt->sizes() != vt->sizes() || kt->size(2) != Hkv || kt->size(3) != D ||
            kt->scalar_type() != at::kBFloat16 || vt->scalar_type() != at::kBFloat16 || !kt->is_contiguous() ||
            !vt->is_contiguous() || !on(kt, dev) || !on(vt, dev) || c.hist_seq->scalar_type() != at::kLong ||
            !c.hist_seq->is_contiguous() || c.hist_seq->numel() < B || !on(c.hist_seq, dev) || c.gbase != 0)
            return 0;
        if (c.hist_slots ? (c.hist_slots->scalar_type() != at::kLong || !c.hist_slots->is_contiguous() ||
                            c.hist_slots->numel() < B || !on(c.hist_slots, dev))
                         : kt->size(0) < B)
            return 0;
    } else if (c.gbase == 0 && kt && vt && c.b_tail) {
        if (kt->dim() != 4) return 0;
        tail = kt->size(1) > 0 && c.max_tail > 0;
        if (tail && (kt->scalar_type() != at::kBFloat16 || vt->scalar_type() != at::kBFloat16 || kt->stride(3) != 1 ||
                     vt->dim() != 4 || vt->stride(3) != 1 || kt->sizes() != vt->sizes() || kt->size(0) < B ||
                     kt->size(2) != Hkv || kt->size(3) != D))
            return 0;
    }
    if (c.err && (c.err->scalar_type() != at::kInt || !on(c.err, dev))) return 0;

    if (c.splits == 0 && c.max_seq < 0) return 0;
    // The serving-recipe kernel keeps three workgroups per compute unit resident with up to 4 q heads per
    // kv head (two with 8, and so do the other kernels); at head_dim 64 one of its waves takes a pair of kv heads.
    const bool plain_planes = gt == 32 && gc == 32 && !scale_bf16 && !v_bf16 && !c.force;
    // K groups of 64 / 128 tokens: the same kernel takes them in pieces of 64 tokens (the plane extents that it
    // addresses are looked at again at the launch; were they too large, the other kernels would serve pieces of groups
    // with the same numbers).
    const bool pieces = gt >= 64 && !scale_bf16 && !v_bf16 && !c.force && D == 128 && R >= 4 && gc >= 32 && !c.bitmap &&
                        (k == 6 || (k == 10 && gt == 128));
    // 64-channel heads with position streams (csrc/ommx_decode_fp32.hip): longer groups in pieces as well
    const bool fp32 = D == 64 && R <= 4 && !c.bitmap && !scale_bf16 && !v_bf16 && !c.force && gt >= 32 && gc >= 32 && k >= 1 &&
                      k <= (gt == 32 ? 6 : 10);
    const int64_t unit = pieces || (fp32 && gt >= 64) ? 64 : gt;           // tokens that a share is made of
    // Longer groups keep two workgroups a compute unit (a third does not fit their LDS, and the shares of a round that is not
    // there made full batches slower than whole groups on the kernel before: 8 x 32 K tokens of 64 x 64 vectors 124 us with
    // three, 113 on that kernel, 95 with two; 32 of 1 to 16 K 134 / 128 / 105; of 128 x 128 with ten outliers 173 / 165 / 125).
    const bool lean = fp32 || (plain_planes && ((D == 128 && R <= 4 && k == 6) ||
                                       (c.bitmap && k >= 1 && k <= 6 && ((D == 128 && R <= 4) ||
                                                                         (D == 64 && R <= 2 && Hkv % 2 == 0)))));
    const bool paired = plain_planes && D == 64 && c.bitmap && k >= 1 && k <= 8 && R <= 4 && Hkv % 2 == 0;
    const int64_t wave_heads = paired ? Hkv / 2 : Hkv;           // waves that one share of the tokens takes

    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    c10::Allocator* const allocator = c10::GetAllocator(c10::DeviceType::CUDA);
    const uint16_t* qp = data<const uint16_t>(c.q);
    auto combine = [&](const float* al, int64_t al_b, int64_t al_h, int64_t al_s, float* lse, int64_t S, const ommx::StateLse* states,
                       const ommx::Shares* dealt) {
        if (hist) {
            const ommx::HistTail t{data<uint16_t>(kt), data<uint16_t>(vt), kt->stride(0), static_cast<int>(kt->size(1)),
                                   data<int64_t>(c.hist_seq), data<int64_t>(c.hist_slots), static_cast<int>(c.ring_sink),
                                   static_cast<int>(c.ring_span), static_cast<int>(c.win_sink), static_cast<int>(c.win_recent)};
            return ommx::decode_combine_hist(al, al_b, al_h, al_s, qp, q.stride(0), q.stride(1), t, data(c.o), o_bf16,
                                             c.o->stride(0), c.o->stride(1), lse, c.lse ? c.lse->stride(0) : Hq, B, Hq,
                                             Hkv, D, S, gt, c.sm_scale, c.cap, *states, dealt, stream);
        }
        return ommx::decode_combine(
            al, al_b, al_h, al_s, qp, q.stride(0), q.stride(1), tail ? data<uint16_t>(kt) : nullptr,
            tail ? data<uint16_t>(vt) : nullptr, tail ? kt->stride(0) : 0, tail ? kt->stride(1) : 0,
            tail ? kt->stride(2) : 0, tail ? vt->stride(0) : 0, tail ? vt->stride(1) : 0, tail ? vt->stride(2) : 0,
            tail ? data<int32_t>(c.b_tail) : nullptr, data<int32_t>(c.seq), data<float>(c.o), c.o->stride(0),
            c.o->stride(1), lse, c.lse->stride(0), B, Hq, Hkv, D, S, gt, tail ? kt->size(1) : 0, c.sm_scale, c.cap,
            states, dealt, stream);
    };
    // The tail rows as states of their own, attended by the last workgroups of the split-KV launch.  Rows must be readable
    // 16 bytes at a time.
    auto rows16 = [&](const at::Tensor* t) {
        return reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0 && t->stride(0) % 8 == 0 && t->stride(1) % 8 == 0 &&
               t->stride(2) % 8 == 0;
    };
    const bool tail_rows = (hist || tail) && !c.ws && !c.force && rows16(kt) && rows16(vt) && B <= 4096 &&
                           (!hist || hist_window_fits(c, gt, kt->size(1)));
    ommx::DecodeTail tl{};
    if (tail_rows) {
        tl = {data<uint16_t>(kt), data<uint16_t>(vt), kt->stride(0), kt->stride(1), kt->stride(2), vt->stride(0),
              vt->stride(1), vt->stride(2), nullptr, static_cast<int>(kt->size(1)), nullptr, nullptr, 0, 0, 0, 0, 0,
              static_cast<int>(gt)};
        if (hist) {
            tl.hist_seq = data<int64_t>(c.hist_seq);
            tl.hist_slots = data<int64_t>(c.hist_slots);
            tl.hist_rows = static_cast<int>(kt->size(1));
            tl.ring_sink = c.ring_span > 0 ? static_cast<int>(c.ring_sink) : 0;
            tl.ring_span = static_cast<int>(c.ring_span);
            tl.win_sink = static_cast<int>(c.win_sink);
            tl.win_recent = static_cast<int>(c.win_recent);
            tl.T = static_cast<int>(c.win_sink + c.win_recent + gt - 1);
        } else {
            tl.tail = data<int32_t>(c.b_tail);
        }
    }
    bool tail_done = false;
    // the merge of either kind: `al` and `states` as the splits have them, `front` slots for the tail before them
    auto merge = [&](float* al, int64_t al_b, int64_t al_h, int64_t al_s, float* lse, int64_t S, const ommx::StateLse& states,
                     const ommx::Shares* dealt) {
        if (!tail_done) return combine(al, al_b, al_h, al_s, lse, S, &states, dealt);
        ommx::StateLse all = states;
        all.p -= ommx::kTailParts * states.s;
        return ommx::fold_states(al - ommx::kTailParts * al_s, al_b, al_h, al_s, all, S + ommx::kTailParts,
                                 ommx::kTailParts + (dealt ? std::min<int>(S, dealt->each) : S), data(c.o), o_bf16,
                                 c.o->stride(0), c.o->stride(1), lse, c.lse ? c.lse->stride(0) : Hq, B, Hq, D, stream);
    };
    // (the argument list that the split-KV entries share; the state strides and the split count come first)
#define OMMX_SPLITKV_ARGS(AL, AL_B, AL_H, AL_S, SPLITS)                                                                  \
    qp, q.stride(0), q.stride(1), data<uint8_t>(c.k_base), data(c.k_scale), data<uint16_t>(c.k_zp),                      \
        own_map ? data<uint16_t>(c.ms) : nullptr, own_map ? data<uint16_t>(c.mc) : nullptr,                              \
        k > 0 ? data<uint8_t>(c.k_index) : nullptr, k > 0 ? data<uint8_t>(c.k_oval) : nullptr, data<uint8_t>(c.v_main),  \
        data(c.v_scale), data<uint16_t>(c.v_zp), data(c.rt), rt.stride(0), data(c.rg), rg.stride(0),                     \
        rt.scalar_type() == at::kLong, data<int32_t>(c.seq), AL, AL_B, AL_H, AL_S, B, Hq, Hkv, D, ps, k,                 \
        c.bitmap ? OMMX_INDEX_BITMAP : OMMX_INDEX_RELIDX7, scale_bf16, gt, gc, v_bf16, SPLITS, c.sm_scale, c.cap, c.off, \
        c.gbase, pages, slots, data<int32_t>(c.err), stream

    // (max_seq bounds how many units there can be; were it too small, the shares would be longer, nothing else)
    const int64_t longest = std::max<int64_t>(1, (c.max_seq + unit - 1) / unit);
    int rc = 1, rc2 = 0;
    const int64_t front = tail_rows ? ommx::kTailParts : 0;
    // the merge inside the launch: its words lie behind the `used` bytes of the scratch, on a line of their own
    const size_t words = static_cast<size_t>(B * wave_heads + 1) * 64;
    auto team_merge = [&](void* scratch, int64_t used, float* lse, int64_t per, bool fused) {
        // (from a number of this process' own on: memory handed on by the driver may hold another one's words)
        static std::atomic<uint64_t> calls{ommx::kFirstCall + (static_cast<uint64_t>(std::random_device{}()) << 14)};
        ommx::TeamMerge m{static_cast<int>(std::min<int64_t>(rt.size(1), INT32_MAX)), static_cast<int>(std::min<int64_t>(rg.size(1), INT32_MAX)),
                          static_cast<int>(per)};
        if (!fused) return m;
        (o_bf16 ? reinterpret_cast<void*&>(m.o16) : reinterpret_cast<void*&>(m.o)) = data(c.o);
        m.o_b = c.o->stride(0); m.o_h = c.o->stride(1);
        m.lse = lse; m.lse_b = c.lse ? c.lse->stride(0) : Hq;
        m.arrivals = reinterpret_cast<unsigned long long*>((reinterpret_cast<uintptr_t>(scratch) + used + 63) / 64 * 64);
        m.number = calls.fetch_add(1, std::memory_order_relaxed);
        return m;
    };
    // the work in equal shares, at most `most` of them for one request
    auto dealt_out = [&](int64_t shares, int64_t few, int64_t singles, int64_t most, bool team, bool fused) {
        const int64_t row = most + front, n = B * Hq * row;
        c10::DataPtr scratch = allocator->allocate(static_cast<size_t>(n * (D + 1) + B * Hq + B) * sizeof(float) + words);
        float *al = static_cast<float*>(scratch.get()), *lse = c.lse ? data<float>(c.lse) : al + n * (D + 1);
        const ommx::StateLse states{al + n * D + front, Hq * row, row, 1};
        const ommx::Shares dealt{static_cast<int>(shares), static_cast<int>(few), static_cast<int>(singles),
                                 static_cast<int>((std::min(shares, B * longest > singles ? B * longest / 2 : shares) + B - 1) / B),
                                 reinterpret_cast<int32_t*>(al + n * (D + 1) + B * Hq)};
        al += front * D;
        const ommx::TeamMerge tm = team_merge(scratch.get(), (n * (D + 1) + B * Hq + B) * 4, lse, 0, fused);
        Py_BEGIN_ALLOW_THREADS
        rc = ommx::decode_splitkv(OMMX_SPLITKV_ARGS(al, Hq * row * D, row * D, D, most), false, &states, &dealt,
                                  tail_rows ? &tl : nullptr, &tail_done, team ? &tm : nullptr);
        if (rc == 0 && !fused) rc2 = merge(al, Hq * row * D, row * D, D, lse, most, states, &dealt);
        Py_END_ALLOW_THREADS
    };
    // S splits of every request
    auto split_up = [&](int64_t S, bool team, int64_t per, bool fused) {
        const int64_t row = S + front, n = B * Hq * row;
        int64_t al_b = Hq * row * D, al_h = row * D, al_s = D;
        c10::DataPtr scratch;
        float *al, *lse = data<float>(c.lse);
        ommx::StateLse states;
        if (c.ws && c.lse) {
            al = c.ws->data_ptr<float>();
            al_b = c.ws->stride(0); al_h = c.ws->stride(1); al_s = c.ws->stride(2);
            states = {al + D, al_b, al_h, al_s};
        } else {
            scratch = allocator->allocate(static_cast<size_t>(n * (D + 1) + B * Hq) * sizeof(float) + words);
            al = static_cast<float*>(scratch.get());
            states = {al + n * D + front, Hq * row, row, 1};
            if (!lse) lse = al + n * (D + 1);
            al += front * D;
        }
        const ommx::TeamMerge tm = team_merge(scratch.get(), (n * (D + 1) + B * Hq) * 4, lse, per, fused);
        Py_BEGIN_ALLOW_THREADS
        rc = ommx::decode_splitkv(OMMX_SPLITKV_ARGS(al, al_b, al_h, al_s, S), c.force, &states, nullptr,
                                  tail_rows ? &tl : nullptr, &tail_done, team ? &tm : nullptr);
        if (rc == 0 && !fused) rc2 = merge(al, al_b, al_h, al_s, lse, S, states, nullptr);
        Py_END_ALLOW_THREADS
    };
    // Short calls: four waves on one kv head of one split (csrc/ommx_decode_team.hip), in 64-token steps, while there are few of
    // those for a compute unit (counted by the longest request).  From there on that kernel's quarter more instructions count: 8 K tokens
    // of 8 kv heads 14.0 us against 14.3, 12 K 17.6 against 15.8; 8 K with 64 q heads 16.6 / 19.8, 16 K 22.8 / 21.3; with 64 channels, whose
    // heads it does not read in pairs of which one is zero, 16 K 13.6 / 18.0, 2 x 12 K (six steps) 15.7 / 17.8; with one kv head, where a
    // workgroup of the other kernel is a single wave, 16 of 1 to 16 K (16 steps) 20.3 / 22.2, but 8 of 20 to 32 K 24.0 / 23.2.
    // Several requests go a step further, their shares being dealt out either way: 3 of 1 to 3.4 K 14.0 / 12.3, 16 of 100 to 620 13.8 / 12.8, 2 x 5 K
    // 15.6 / 14.7, 16 x 600 16.0 / 15.4 (the other kernel's time first), 6 of 200 to 1600 with 64 q heads 14.5 / 13.3.  Not where the
    // workgroups of their tails crowd the ones of the shares: 24 of 40 to 400 13.2 / 13.7, 48 of 40 to 300 16.2 / 19.8, 8 x 1250
    // with 64 q heads 18.3 / 19.6.  (At six and eight steps ragged batches still gain, 4 of 1 to 4 K 16.3 / 14.9, and equal ones lose, 24 of 1.0 to
    // 1.4 K with 4 heads 17.1 / 18.7; how long they are beside the longest is not known here.)
    // (a range of groups without a tail, of which the caller merges the states, has the rounding of the whole then)
    const bool no_tail = !hist && !tail && !c.ws && !c.force;
    if (c.splits == 0 && (tail_rows || no_tail) && plain_planes && k == 6 && B <= 64 && (D == 128 || paired)) {
        const int64_t cus = cu_count(dev.index()), steps = (longest + 1) / 2, all = B * steps * wave_heads;
        const bool few = B > 1 && B * wave_heads * (R <= 4 ? 4 : 10) <= 2 * cus;
        if (all <= cus * (paired || wave_heads == 1 ? 8 : few ? 5 : 4)) {
            // The merge inside the launch while its one workgroup has little to read, instead of a launch of its own (3.5 us of host
            // time; 1 K tokens 8.5 us against 9.1 to 10).  Not under capture: see TeamMerge.
            hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
            const bool eager = hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
            // Nor where a result lies in what the call reads: the last workgroup of one head writes it while those of others still read.
            auto apart = [&] {
                const Span o(*c.o), lse = c.lse ? Span(*c.lse) : o;
                for (const at::Tensor* t : {c.q, c.k_base, c.k_scale, c.k_zp, c.k_index, c.k_oval, c.v_main, c.v_scale, c.v_zp, c.ms, c.mc, c.k_tail,
                                            c.v_tail, c.b_tail, c.hist_seq, c.hist_slots, c.rt, c.rg, c.seq}) {
                    if (!t) continue;
                    const Span in(*t);
                    if (in.meets(o) || in.meets(lse)) return false;
                }
                return true;
            };
            auto merged = [&](int64_t states) {
                return eager && states <= ommx::kTeamMerged && states * (Hq / wave_heads) * D <= ommx::kTeamMerged * 512 && apart();
            };
            // one request: up to three workgroups a compute unit (two with 8 heads); several: two, or a split a step where all of those fit
            const int64_t room = std::clamp<int64_t>((B == 1 && R <= 4 ? 3 : 2) * cus / wave_heads, 1, 508);
            if (B == 1 || B * steps <= room) {
                const int64_t each = (steps + room - 1) / room, S = (steps + each - 1) / each;
                split_up(S, true, 2 * each, merged(S));
            } else if (B <= room) {
                const int64_t most = std::min<int64_t>({508, steps, std::max<int64_t>(8, 4 * room / B)});
                dealt_out(room, room, 0, most, true, merged(most));
            }
        }
    }
    if (rc == 1 && c.splits == 0 && !c.ws && !c.force && B > 1) {
        // Several requests and nobody asked for a split count: the kernels deal the groups out in equal shares, as many
        // as are resident at once (a wave per kv head and share).  One request gets at most 256 of them (its states
        // are merged on chip), 64 with many (request, head) pairs, where the combine's small form serves, and no
        // more than four times its even part, which bounds the workspace.
        const int64_t fit = cu_count(dev.index()) * 4 / wave_heads;
        const int64_t shares = std::min({int64_t{2048}, fit * (lean ? 3 : 2), B * longest});
        const int64_t few = std::min(shares, fit * 2);
        const int64_t most = std::min({int64_t{B * Hq >= 256 ? 64 : (shares > 256 * B && longest > 512 ? 512 : 256)}, longest,
                                       std::max<int64_t>(8, 4 * shares / B)});
        // A batch that cannot have more groups than SIMDs is left to fixed splits of one group: those need not find their
        // share (0.3 us).  From there on a split per group of the longest request would put two workgroups on some
        // compute units, empty ones among them: 8 requests of 97 to 701 tokens 9.9 us as 23 splits each, 8.5 dealt out.
        if (few >= B && B * longest > fit) dealt_out(shares, few, paired ? 2 * fit : fit, most, false, false);
    }
    if (rc == 1) {
        int64_t S = c.splits;
        if (S == 0) {
            S = auto_splits(c.max_seq, B, wave_heads, cu_count(dev.index()), unit, c.mean, lean ? 3 : 2);
            // What this kernel likes best can be more than the public rule gives for the recipe's own groups and heads, by which a
            // caller sizes its workspace (128-token groups, 8 kv heads, 4096 tokens: 64 against 32): that many then.
            if (c.ws && c.ws->dim() == 4 && c.ws->size(2) < S)
                S = std::min<int64_t>(S, auto_splits(c.max_seq, B, Hkv, cu_count(dev.index()), gt, c.mean, 2));
        }
        if (c.ws && (c.ws->scalar_type() != at::kFloat || c.ws->dim() != 4 || c.ws->size(0) != B || c.ws->size(1) != Hq ||
                     c.ws->size(2) < S || c.ws->size(3) < D + 1 || c.ws->stride(3) != 1))
            return 0;
        split_up(S, false, 0, false);
    }
#undef OMMX_SPLITKV_ARGS
    if (failed(rc, "ommx_decode_splitkv") || failed(rc2, "ommx_decode_combine")) return -1;
    written(*c.o);
    if (c.lse) written(*c.lse);
    return 1;
}

PyObject* answer(int rc) {
    if (rc < 0) return nullptr;
    return PyBool_FromLong(rc);
}

// (a, b, heads, head_dim): whether both are [rows, heads, head_dim]
PyObject* py_rows_fit(PyObject*, PyObject* const* a, Py_ssize_t n) {
    bool ok = n == 4;
    const at::Tensor *x = ok ? as_tensor(a[0], ok) : nullptr, *y = ok ? as_tensor(a[1], ok) : nullptr;
    if (!ok) { PyErr_SetString(PyExc_TypeError, "rows_fit: two tensors, heads and head_dim expected"); return nullptr; }
    const int64_t H = as_int(a[2], ok), D = as_int(a[3], ok);
    auto fits = [&](const at::Tensor& t) {
        return !t.unsafeGetTensorImpl()->has_symbolic_sizes_strides() && t.dim() == 3 && t.size(1) == H && t.size(2) == D;
    };
    return PyBool_FromLong(ok && fits(*x) && fits(*y));
}

// (tensors or None ...)
PyObject* py_plain(PyObject*, PyObject* const* a, Py_ssize_t n) { return PyBool_FromLong(plain_call(a, n)); }

// The arguments of ommx_paged_decode_attention_canonical, in the order of DecodeArg.
PyObject* py_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != A_COUNT) { PyErr_SetString(PyExc_TypeError, "decode: wrong number of arguments"); return nullptr; }
    bool ok = true;
    DecodeCall c;
    c.q = as_tensor(a[A_Q], ok); c.k_base = as_tensor(a[A_KBASE], ok); c.k_scale = as_tensor(a[A_KSCALE], ok);
    c.k_zp = as_tensor(a[A_KZP], ok); c.k_oval = as_tensor_or_none(a[A_KOVAL], ok);
    c.v_main = as_tensor(a[A_VMAIN], ok); c.v_scale = as_tensor(a[A_VSCALE], ok); c.v_zp = as_tensor(a[A_VZP], ok);
    c.k_tail = as_tensor_or_none(a[A_KTAIL], ok); c.v_tail = as_tensor_or_none(a[A_VTAIL], ok);
    c.b_tail = as_tensor_or_none(a[A_BTAIL], ok); c.o = as_tensor(a[A_O], ok); c.lse = as_tensor(a[A_LSE], ok);
    c.rt = as_tensor(a[A_RT], ok); c.rg = as_tensor(a[A_RG], ok); c.seq = as_tensor(a[A_SEQ], ok);
    c.ms = as_tensor_or_none(a[A_MS], ok); c.mc = as_tensor_or_none(a[A_MC], ok);
    c.ws = as_tensor_or_none(a[A_WS], ok); c.err = as_tensor_or_none(a[A_ERR], ok);
    c.sm_scale = as_double(a[A_SM], ok); c.cap = as_double(a[A_CAP], ok);
    c.ps = as_int(a[A_PS], ok); c.k = as_int(a[A_KOUT], ok); c.off = as_int(a[A_OFF], ok); c.gbase = as_int(a[A_GBASE], ok);
    c.bitmap = as_bool(a[A_BITMAP], ok); c.int8 = as_bool(a[A_INT8], ok); c.force = as_bool(a[A_FORCE], ok);
    c.want_map = as_bool(a[A_MAP], ok);
    if (a[A_SPLITS] != Py_None) {
        c.splits = as_int(a[A_SPLITS], ok);
        if (c.splits < 1) ok = false;
    }
    if (a[A_MAXSEQ] != Py_None) c.max_seq = std::max<int64_t>(1, as_int(a[A_MAXSEQ], ok));
    if (a[A_MAXTAIL] != Py_None) c.max_tail = as_int(a[A_MAXTAIL], ok);
    if (a[A_MEAN] != Py_None) c.mean = as_double(a[A_MEAN], ok);
    c.k_index = as_tensor_or_none(a[c.bitmap ? A_KOBMP : A_KOIDX], ok);
    const bool combinadic = as_bool(a[A_COMBI], ok);
    if (!ok || combinadic || (!is_word(a[A_KFMT], "i2f4") && !is_word(a[A_KFMT], "itf4"))) Py_RETURN_FALSE;
    return answer(run_decode(c));
}

// ── stores ─────────────────────────────────────────────────────────────────────────────────────

bool is_index(const at::Tensor* t, c10::Device dev, at::ScalarType type, int64_t n) {
    return !t || (t->scalar_type() == type && t->is_contiguous() && t->numel() >= n && t->device() == dev);
}

// [T, H, D] rows of bf16 or fp32 with a contiguous last axis
bool is_rows(const at::Tensor& t) {
    return t.dim() == 3 && (t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat) && t.stride(2) == 1;
}

struct Recipe {
    int64_t k, gt, gc;
    bool bitmap, abs, v_bf16;
    int mode;
};
// (outliers, group_tokens, group_channels, outlier_repr, outlier_select, use_pow2, kv_int8_scale, v_format)
bool read_recipe(PyObject* const* a, Recipe& r) {
    bool ok = true;
    r.k = as_int(a[0], ok); r.gt = as_int(a[1], ok); r.gc = as_int(a[2], ok);
    r.bitmap = is_word(a[3], "bitmap");
    if (!r.bitmap && !is_word(a[3], "relidx7")) return false;
    r.abs = is_word(a[4], "abs");
    if (!r.abs && !is_word(a[4], "signed")) return false;
    const bool pow2 = as_bool(a[5], ok), int8 = as_bool(a[6], ok);
    r.mode = !pow2 ? OMMX_SCALE_BF16 : (int8 ? OMMX_SCALE_POW2_INT8 : OMMX_SCALE_POW2_BF16);
    r.v_bf16 = is_word(a[7], "bf16");
    if (!r.v_bf16 && !is_word(a[7], "i2")) return false;
    return ok && r.k >= 0 && r.k <= 16 && is_group_size(r.gt) && is_group_size(r.gc);
}

struct Planes {
    const at::Tensor *k_base = nullptr, *k_scale = nullptr, *k_zp = nullptr, *ms = nullptr, *mc = nullptr,
                     *index = nullptr, *oval = nullptr, *v_main = nullptr, *v_scale = nullptr, *v_zp = nullptr;
};
PyObject* g_names[11];      // interned keys of a plane dict
PyObject* g_bitmap;
enum { N_KBASE, N_KSCALE, N_KZP, N_MS, N_MC, N_OBMP, N_OIDX, N_OVAL, N_VMAIN, N_VSCALE, N_VZP };

bool read_planes(PyObject* d, const Recipe& r, Planes& p) {
    if (!PyDict_Check(d)) return false;
    bool ok = true;
    auto get = [&](int name) -> const at::Tensor* {
        PyObject* o = PyDict_GetItem(d, g_names[name]);      // borrowed
        return !o || o == Py_None ? nullptr : as_tensor(o, ok);
    };
    p = {get(N_KBASE), get(N_KSCALE), get(N_KZP), get(N_MS), get(N_MC), get(r.bitmap ? N_OBMP : N_OIDX),
         get(N_OVAL), get(N_VMAIN), get(N_VSCALE), get(N_VZP)};
    if (!ok || !p.k_base || !p.k_scale || !p.k_zp || !p.v_main || !p.v_scale || !p.v_zp) return false;
    if (r.k > 0 && (!p.index || p.index->dim() < 1 ||
                    p.index->size(-1) != (r.bitmap ? (r.gt + 7) / 8 : (7 * r.k + 7) / 8)))
        return false;
    const at::ScalarType step = r.mode == OMMX_SCALE_POW2_INT8 ? at::kChar : at::kBFloat16;
    return (p.v_main->scalar_type() == at::kBFloat16) == r.v_bf16 && p.k_scale->scalar_type() == step &&
           p.v_scale->scalar_type() == step;
}

int launch_store(const at::Tensor& K, const at::Tensor& V, int64_t row0, const Planes& p, const Recipe& r, int64_t T, int64_t ps,
                 const int32_t* src, const int32_t* pages, const int32_t* groups, const at::Tensor& table,
                 int32_t* err, const ommx::StoreExtras& extras, hipStream_t stream) {
    auto from = [row0](const at::Tensor& t) {
        return static_cast<const char*>(t.data_ptr()) + row0 * t.stride(0) * static_cast<int64_t>(t.element_size());
    };
    return ommx::store_pack(
        from(K), from(V), K.scalar_type() == at::kFloat, K.stride(0), K.stride(1), V.stride(0), V.stride(1),
        src, T, K.size(1), K.size(2), ps, r.k, r.bitmap ? OMMX_INDEX_BITMAP : OMMX_INDEX_RELIDX7, r.abs, r.mode, r.gt,
        r.gc, r.v_bf16, pages, groups, table.data_ptr<float>(), data<uint8_t>(p.k_base), data(p.k_scale),
        data<uint16_t>(p.k_zp), data<uint16_t>(p.ms), data<uint16_t>(p.mc), data<uint8_t>(p.index),
        data<uint8_t>(p.oval), data<uint8_t>(p.v_main), data(p.v_scale), data<uint16_t>(p.v_zp), err, extras, stream);
}

// Groups of a pool's history (contiguous, [slots, rows, heads, head_dim]) as arguments of one store launch, where its kernel takes
// them: 1 with nothing done otherwise.  Rows that turn around at most once.
int launch_ring_groups(const at::Tensor& kh, const at::Tensor& vh, const std::vector<int64_t>& pairs, const Planes& p, const Recipe& r, int64_t ps,
                       int64_t sink, int64_t span, int64_t wsink, int64_t per_seq, const at::Tensor& table, int32_t* err,
                       const ommx::StepWrite* step, hipStream_t stream) {
    const int64_t count = static_cast<int64_t>(pairs.size()) / 2, N = kh.size(0), rows = kh.size(1), H = kh.size(2), D = kh.size(3);
    if (count > ommx::kRingGroups || N * rows > INT32_MAX || N * per_seq > INT32_MAX || (span != 0 && (wsink < sink || span < r.gt))) return 1;
    ommx::RingGroups ring;
    for (int64_t i = 0; i < count; ++i) {
        const int64_t pos = wsink + pairs[2 * i + 1] * r.gt, slot = span > 0 ? sink + (pos - sink) % span : pos;
        ring.of[i] = {static_cast<int32_t>(pairs[2 * i] * rows + slot), span > 0 ? static_cast<int32_t>(sink + span - slot) : INT32_MAX,
                      static_cast<int32_t>(pairs[2 * i] * per_seq + pairs[2 * i + 1])};
    }
    ommx::StoreExtras extras;
    extras.ring = &ring;
    extras.ring_span = static_cast<int>(span);
    extras.step = step;
    return ommx::store_pack(
        kh.data_ptr(), vh.data_ptr(), 0, H * D, D, H * D, D, nullptr, count * r.gt, H, D, ps, r.k, r.bitmap ? OMMX_INDEX_BITMAP : OMMX_INDEX_RELIDX7,
        r.abs, r.mode, r.gt, r.gc, r.v_bf16, nullptr, nullptr, table.data_ptr<float>(), data<uint8_t>(p.k_base), data(p.k_scale),
        data<uint16_t>(p.k_zp), data<uint16_t>(p.ms), data<uint16_t>(p.mc), data<uint8_t>(p.index), data<uint8_t>(p.oval),
        data<uint8_t>(p.v_main), data(p.v_scale), data<uint16_t>(p.v_zp), err, extras, stream);
}

bool is_history(const at::Tensor& k, const at::Tensor& v) {
    return k.dim() == 4 && k.sizes() == v.sizes() && k.scalar_type() == at::kBFloat16 &&
           v.scalar_type() == at::kBFloat16 && k.is_contiguous() && v.is_contiguous() && k.is_cuda();
}

// (k_hist, v_hist, req, n_head, lo, sink, span) at `a`: rows [0, n_head) and [lo, T) of K / V into a request's history
bool read_block_rows(const at::Tensor& K, const at::Tensor& V, PyObject* const* a, int64_t pos0, ommx::BlockRows& out) {
    bool ok = true;
    const at::Tensor *kh = as_tensor(a[0], ok), *vh = as_tensor(a[1], ok);
    const int64_t req = as_int(a[2], ok), head = as_int(a[3], ok), lo = as_int(a[4], ok), sink = as_int(a[5], ok),
                  span = as_int(a[6], ok);
    if (!ok || !is_history(*kh, *vh) || !is_rows(K) || !is_rows(V) || K.sizes() != V.sizes() ||
        K.device() != kh->device() || V.device() != kh->device())
        return false;
    const int64_t T = K.size(0), rows = kh->size(1), H = kh->size(2), D = kh->size(3);
    // every slot has to lie inside the history: below the ring's end, or the block's last position without a ring
    if (K.size(1) != H || K.size(2) != D || D % 8 || req < 0 || req >= kh->size(0) || pos0 < 0 || head < 0 ||
        lo < head || lo > T || sink < 0 || span < 0 || (span > 0 ? sink + span : pos0 + T) > rows)
        return false;
    out = ommx::block_rows(K.data_ptr(), V.data_ptr(), K.scalar_type() == at::kFloat, V.scalar_type() == at::kFloat,
                           K.stride(0), K.stride(1), V.stride(0), V.stride(1),
                           data<uint16_t>(kh) + req * kh->stride(0), data<uint16_t>(vh) + req * vh->stride(0), pos0,
                           head, lo, T, H, D, sink, span);
    return true;
}

// (K, V, planes, page_size, src_rows, dst_pages, dst_groups, err_flag, num_tokens, table, row0, page0, group0, recipe x 8);
// without src_rows the tokens are the rows row0, row0 + 1, ...; the tables are read from entry page0 / group0 on
// Seven more arguments (see read_block_rows): rows of the same bf16 block copied into a request's history by the same launch.
PyObject* py_store_pack(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 21 && n != 28) { PyErr_SetString(PyExc_TypeError, "store_pack: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *K = as_tensor(a[0], ok), *V = as_tensor(a[1], ok), *src = as_tensor_or_none(a[4], ok),
                     *pages = as_tensor_or_none(a[5], ok), *groups = as_tensor_or_none(a[6], ok),
                     *err = as_tensor_or_none(a[7], ok), *table = as_tensor(a[9], ok);
    const int64_t ps = as_int(a[3], ok), row0 = as_int(a[10], ok), page0 = as_int(a[11], ok), group0 = as_int(a[12], ok);
    Recipe r;
    Planes p;
    if (!ok || !read_recipe(a + 13, r) || !read_planes(a[2], r, p) || !is_rows(*K) || !is_rows(*V) || ps < 1 ||
        K->scalar_type() != V->scalar_type() || K->device() != V->device() || !K->is_cuda())
        Py_RETURN_FALSE;
    const c10::Device dev = K->device();
    const int64_t T = a[8] != Py_None ? as_int(a[8], ok) : (src ? src->numel() : K->size(0));
    if (!ok || T < 0 || row0 < 0 || page0 < 0 || group0 < 0 || (!src && row0 + T > K->size(0)) ||
        !is_index(src, dev, at::kInt, T) || !is_index(pages, dev, at::kInt, page0 + T / ps) ||
        !is_index(groups, dev, at::kInt, group0 + T / r.gt))
        Py_RETURN_FALSE;
    ommx::StoreExtras extras;
    ommx::BlockRows rows;
    if (n == 28) {
        // (rows that come out of the history itself: not while it is being written)
        if (T == 0 || K->scalar_type() != at::kBFloat16 || !read_block_rows(*K, *V, a + 21, 0, rows) ||
            rows.rows > ommx::kRowSlices * (T / r.gt))
            Py_RETURN_FALSE;
        for (PyObject* hist : {a[21], a[22]})
            if (K->is_alias_of(THPVariable_Unpack(hist)) || V->is_alias_of(THPVariable_Unpack(hist))) Py_RETURN_FALSE;
        extras.rows = &rows;
    }
    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = launch_store(*K, *V, row0, p, r, T, ps, data<int32_t>(src), pages ? data<int32_t>(pages) + page0 : nullptr,
                      groups ? data<int32_t>(groups) + group0 : nullptr, *table, data<int32_t>(err), extras, stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "ommx_store_pack")) return nullptr;
    Py_RETURN_TRUE;
}

// Host-visible error words of block packing, OMMX_STORE_ERR_WORDS ints each.  A call takes a block and gives it back
// when it has been read; at most kKeptFlags idle ones are kept (more go back to torch's pinned allocator).
constexpr size_t kKeptFlags = 16;
struct FlagPool {
    std::mutex lock;
    std::vector<at::Tensor> idle;
};
FlagPool& flag_pool() {
    static FlagPool* const pool = new FlagPool;      // never destroyed: the runtime may be gone before static destructors
    return *pool;
}
at::Tensor take_flags() {
    at::Tensor t;
    {
        FlagPool& pool = flag_pool();
        std::lock_guard<std::mutex> hold(pool.lock);
        if (!pool.idle.empty()) { t = std::move(pool.idle.back()); pool.idle.pop_back(); }
    }
    if (!t.defined()) t = at::empty({OMMX_STORE_ERR_WORDS}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    std::fill_n(t.data_ptr<int32_t>(), OMMX_STORE_ERR_WORDS, 0);
    return t;
}

// A block packed into planes of its own with identity tables: the launch is under way when this returns; `t` takes the planes and the
// error words.  0 launched, 1 not for this path (nothing done), -1 failed.
enum { FLAGS, KBASE, KSCALE, KZP, INDEX, OVAL, MS, MC, VMAIN, VSCALE, VZP, TOK, GRP, COUNT };
int launch_block(const at::Tensor& K, const at::Tensor& V, int64_t ps, bool own_map, const at::Tensor& table, const Recipe& r,
                 hipStream_t stream, at::Tensor (&t)[COUNT]) {
    const int64_t T = K.size(0), H = K.size(1), D = K.size(2), G = T / r.gt, P = T / ps;
    c10::Allocator* const allocator = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
    // (a dozen tensors: their memory from the allocator directly, the dispatcher would cost a microsecond for each, and what holds it
    // is made while the kernel runs)
    struct Part {
        int64_t shape[4];
        int dims;
        at::ScalarType type;
        size_t bytes = 0;
        c10::DataPtr mem;
    } part[COUNT];
    auto make = [&](int i, std::initializer_list<int64_t> shape, at::ScalarType type) {
        Part& x = part[i];
        std::copy(shape.begin(), shape.end(), x.shape);
        x.dims = static_cast<int>(shape.size());
        x.type = type;
        x.bytes = c10::elementSize(type);
        for (int64_t n : shape) x.bytes *= static_cast<size_t>(n);
        x.mem = allocator->allocate(x.bytes);
        return x.mem.get();
    };
    const at::ScalarType step = r.mode == OMMX_SCALE_POW2_INT8 ? at::kChar : at::kBFloat16;
    t[FLAGS] = take_flags();
    void *index = nullptr, *oval = nullptr, *ms = nullptr, *mc = nullptr;
    void* const k_base = make(KBASE, {P, ps, H, D / 4}, at::kByte);
    void* const k_scale = make(KSCALE, {G, H, D}, step);
    void* const k_zp = make(KZP, {G, H, D}, at::kBFloat16);
    if (r.k > 0) {
        index = make(INDEX, {G, H, D, r.bitmap ? (r.gt + 7) / 8 : (7 * r.k + 7) / 8}, at::kByte);
        oval = make(OVAL, {G, H, D, (r.k + 1) / 2}, at::kByte);
        if (own_map) {
            ms = make(MS, {G, H, D}, at::kBFloat16);
            mc = make(MC, {G, H, D}, at::kBFloat16);
        }
    }
    void* const v_main = r.v_bf16 ? make(VMAIN, {P, ps, H, D}, at::kBFloat16) : make(VMAIN, {P, ps, H, D / 4}, at::kByte);
    void* const v_scale = make(VSCALE, {P, ps, H, D / r.gc}, step);
    void* const v_zp = make(VZP, {P, ps, H, D / r.gc}, at::kBFloat16);
    void* const tok = make(TOK, {1, P}, at::kInt);
    void* const grp = make(GRP, {1, G}, at::kInt);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ommx::store_pack(K.data_ptr(), V.data_ptr(), K.scalar_type() == at::kFloat, K.stride(0), K.stride(1), V.stride(0), V.stride(1),
                          nullptr, T, H, D, ps, r.k, r.bitmap ? OMMX_INDEX_BITMAP : OMMX_INDEX_RELIDX7, r.abs, r.mode, r.gt, r.gc, r.v_bf16,
                          nullptr, nullptr, table.data_ptr<float>(), static_cast<uint8_t*>(k_base), k_scale, static_cast<uint16_t*>(k_zp),
                          static_cast<uint16_t*>(ms), static_cast<uint16_t*>(mc), static_cast<uint8_t*>(index), static_cast<uint8_t*>(oval),
                          static_cast<uint8_t*>(v_main), v_scale, static_cast<uint16_t*>(v_zp), t[FLAGS].data_ptr<int32_t>(),
                          {true, static_cast<int32_t*>(tok), static_cast<int32_t*>(grp)}, stream);
    Py_END_ALLOW_THREADS
    for (int i = 0; i < COUNT; ++i) {
        Part& x = part[i];
        if (x.bytes == 0) continue;
        t[i] = at::detail::make_tensor_base<c10::TensorImpl>(
            c10::make_intrusive<c10::StorageImpl>(c10::StorageImpl::use_byte_size_t(), x.bytes, std::move(x.mem), allocator, true),
            c10::DispatchKeySet(c10::DispatchKey::CUDA), c10::scalarTypeToTypeMeta(x.type));
        t[i].unsafeGetTensorImpl()->generic_set_sizes_contiguous(at::IntArrayRef(x.shape, x.dims));
    }
    return rc;
}
// Should nobody ask for the errors of a block, its words must not be handed on before the kernel is through with them.
void keep_flags_for(const at::Tensor& flags, c10::Device dev) {
    at::getHostAllocator(c10::DeviceType::CUDA)->record_event(flags.data_ptr(), flags.storage().data_ptr().get_context(),
                                                              c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).unwrap());
}
// The error bits, once the launch has ended; the words go back to those kept idle.
long take_errors(const at::Tensor& flags) {
    const int32_t* words = flags.data_ptr<int32_t>();
    long bits = 0;
    for (int i = 0; i < OMMX_STORE_ERR_WORDS; ++i) bits |= (words[i] ? 1L : 0L) << i;
    FlagPool& pool = flag_pool();
    std::lock_guard<std::mutex> hold(pool.lock);
    if (pool.idle.size() < kKeptFlags) pool.idle.push_back(flags);
    return bits;
}
bool is_block(const at::Tensor& K, const at::Tensor& V, int64_t ps, const Recipe& r) {
    return is_rows(K) && is_rows(V) && K.sizes() == V.sizes() && ps >= 1 && K.scalar_type() == V.scalar_type() &&
           K.device() == V.device() && K.is_cuda() && K.size(0) >= 1 && K.size(0) % ps == 0 && K.size(0) % r.gt == 0 && K.size(2) % r.gc == 0;
}

// (K, V, page_size, kv_outlier_map, table, recipe x 8) -> (flags, k_base, k_scale, k_zp, k_index, k_oval, k_mapscale,
// k_mapcenter, v_main, v_scale, v_zp, req_to_token, req_to_group), or False.  Launches the packing of a block into planes
// of its own with identity tables.  The caller does its own work and then asks block_errors(flags), the one host
// stop: the error bits come back through host memory that the kernel writes only when there is something to
// report, so nothing is copied.
PyObject* py_pack_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 13) { PyErr_SetString(PyExc_TypeError, "pack_block: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *K = as_tensor(a[0], ok), *V = as_tensor(a[1], ok), *table = as_tensor(a[4], ok);
    const int64_t ps = as_int(a[2], ok);
    const bool own_map = as_bool(a[3], ok);
    Recipe r;
    if (!ok || !read_recipe(a + 5, r) || !is_block(*K, *V, ps, r)) Py_RETURN_FALSE;
    const c10::Device dev = K->device();
    c10::hip::HIPGuard guard(dev.index());
    at::Tensor t[COUNT];
    const int rc = launch_block(*K, *V, ps, own_map, *table, r, stream_of(dev), t);
    keep_flags_for(t[FLAGS], dev);
    if (failed(rc, "ommx_store_pack")) return nullptr;
    PyObject* out = PyTuple_New(COUNT);
    for (int i = 0; i < COUNT; ++i) {
        if (!t[i].defined()) { Py_INCREF(Py_None); PyTuple_SET_ITEM(out, i, Py_None); }
        else PyTuple_SET_ITEM(out, i, THPVariable_Wrap(std::move(t[i])));
    }
    return out;
}

// The whole of a block's call for arguments in their plain form: (K, V, table, page_size, device, kv_outlier_map, k_format, outliers,
// group_tokens, group_channels, outlier_repr, outlier_select, use_pow2, kv_int8_scale, v_format), None for either flag that may be
// left out.  -> the plane dict, the error bits of a block that has any, or False with nothing done.
constexpr const char* kBlockKeys[] = {
    "k_base", "k_scale", "k_zp", "k_oidx", "k_oval", "k_crank", "k_obmp", "k_fp4_mapscale", "k_fp4_mapcenter", "k_field_bytes",
    "v_main", "v_scale", "v_zp", "req_to_token", "req_to_group", "head_dim", "n_kv_heads", "num_tokens", "n_groups", "page_size",
    "outliers_per_vector", "outlier_repr", "outlier_select", "group_tokens", "group_channels", "k_format", "v_format", "k_base_bits",
    "oval_bits", "use_pow2", "kv_outlier_map", "kv_int8_scale"};
constexpr int kBlockKeyCount = sizeof(kBlockKeys) / sizeof(kBlockKeys[0]);
PyObject* g_block_keys[kBlockKeyCount];

PyObject* py_pack_whole_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 15) { PyErr_SetString(PyExc_TypeError, "pack_whole_block: wrong number of arguments"); return nullptr; }
    if (!plain_call(a, 2)) Py_RETURN_FALSE;
    bool ok = true;
    const at::Tensor *K = as_tensor(a[0], ok), *V = as_tensor(a[1], ok), *table = as_tensor(a[2], ok);
    const int64_t ps = as_int(a[3], ok);
    PyObject* const recipe[8] = {a[7], a[8], a[9], a[10], a[11], a[12], a[13] == Py_None ? Py_True : a[13], a[14]};
    const bool map = a[5] == Py_None || as_bool(a[5], ok);
    Recipe r;
    if (!ok || !(is_word(a[6], "i2f4") || is_word(a[6], "itf4")) || !read_recipe(recipe, r) || !is_block(*K, *V, ps, r) ||
        K->size(2) % 32 || K->size(2) > 256 || r.k > r.gt)
        Py_RETURN_FALSE;
    const c10::Device dev = K->device();
    if (THPDevice_Check(a[4])) {
        const c10::Device& want = reinterpret_cast<THPDevice*>(a[4])->device;
        if (!want.is_cuda() || (want.has_index() ? want.index() : c10::hip::current_device()) != dev.index()) Py_RETURN_FALSE;
    } else if (!is_word(a[4], "cuda") || c10::hip::current_device() != dev.index()) {
        Py_RETURN_FALSE;
    }
    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    at::Tensor t[COUNT];
    if (failed(launch_block(*K, *V, ps, map, *table, r, stream, t), "ommx_store_pack")) { keep_flags_for(t[FLAGS], dev); return nullptr; }
    // (put together while the kernel runs)
    const at::Tensor flags = t[FLAGS];
    PyObject* const out = PyDict_New();
    int key = 0;
    bool good = out != nullptr;
    auto put = [&](PyObject* value) {          // takes the reference
        good = good && value && PyDict_SetItem(out, g_block_keys[key], value) == 0;
        ++key;
        Py_XDECREF(value);
    };
    auto tensor = [&](int i) { put(t[i].defined() ? THPVariable_Wrap(std::move(t[i])) : Py_NewRef(Py_None)); };
    auto none = [&]() { put(Py_NewRef(Py_None)); };
    auto number = [&](int64_t v) { put(PyLong_FromLongLong(v)); };
    auto flag = [&](bool v) { put(Py_NewRef(v ? Py_True : Py_False)); };
    auto same = [&](PyObject* o) { put(Py_NewRef(o)); };
    const int64_t T = K->size(0);
    tensor(KBASE); tensor(KSCALE); tensor(KZP);
    if (r.bitmap) none(); else tensor(INDEX);
    tensor(OVAL); none();
    if (r.bitmap) tensor(INDEX); else none();
    tensor(MS); tensor(MC);
    number(r.bitmap && r.k > 0 ? (r.gt + 7) / 8 : 0);
    tensor(VMAIN); tensor(VSCALE); tensor(VZP); tensor(TOK); tensor(GRP);
    number(K->size(2)); number(K->size(1)); number(T); number(T / r.gt); number(ps); number(r.k);
    same(recipe[3]); same(recipe[4]); number(r.gt); number(r.gc); same(a[6]); same(recipe[7]);
    number(2); number(4);
    flag(recipe[5] == Py_True); flag(map && r.k > 0); flag(recipe[5] == Py_True && recipe[6] == Py_True);
    hipError_t waited;
    Py_BEGIN_ALLOW_THREADS
    waited = hipStreamSynchronize(stream);
    Py_END_ALLOW_THREADS
    if (waited != hipSuccess) {
        keep_flags_for(flags, dev);
        Py_XDECREF(out);
        PyErr_Format(PyExc_RuntimeError, "ommx_store_pack: %s", hipGetErrorString(waited));
        return nullptr;
    }
    const long bits = take_errors(flags) & ~static_cast<long>(OMMX_NOTE_WIDE_STEP);
    if (good && bits == 0) return out;
    Py_XDECREF(out);
    return good ? PyLong_FromLong(bits) : nullptr;
}

// (flags, tensor of the packing device): waits for the current stream of that device and returns the error bits
PyObject* py_block_errors(PyObject*, PyObject* const* a, Py_ssize_t n) {
    bool ok = n == 2;
    const at::Tensor *flags = ok ? as_tensor(a[0], ok) : nullptr, *on_dev = ok ? as_tensor(a[1], ok) : nullptr;
    if (!ok || flags->numel() != OMMX_STORE_ERR_WORDS || flags->scalar_type() != at::kInt || !on_dev->is_cuda()) {
        PyErr_SetString(PyExc_TypeError, "block_errors: flags of pack_block and a GPU tensor expected");
        return nullptr;
    }
    c10::hip::HIPGuard guard(on_dev->device().index());
    hipStream_t stream = stream_of(on_dev->device());
    hipError_t waited;
    Py_BEGIN_ALLOW_THREADS
    waited = hipStreamSynchronize(stream);
    Py_END_ALLOW_THREADS
    if (waited != hipSuccess) {
        PyErr_Format(PyExc_RuntimeError, "ommx_store_pack: %s", hipGetErrorString(waited));
        return nullptr;
    }
    return PyLong_FromLong(take_errors(*flags));
}

// ── bf16 row history ───────────────────────────────────────────────────────────────────────────

// (k_hist, v_hist, pos, k, v, sink, span, slots, pos_next, err_flag)
PyObject* py_ring_write(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 10) { PyErr_SetString(PyExc_TypeError, "ring_write: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *kh = as_tensor(a[0], ok), *vh = as_tensor(a[1], ok), *pos = as_tensor(a[2], ok),
                     *k = as_tensor(a[3], ok), *v = as_tensor(a[4], ok), *slots = as_tensor_or_none(a[7], ok),
                     *next = as_tensor_or_none(a[8], ok), *err = as_tensor_or_none(a[9], ok);
    const int64_t sink = as_int(a[5], ok), span = as_int(a[6], ok);
    if (!ok || !is_history(*kh, *vh) || k->dim() != 3 || k->sizes() != v->sizes()) Py_RETURN_FALSE;
    const c10::Device dev = kh->device();
    const int64_t B = k->size(0), N = kh->size(0), rows = kh->size(1), H = kh->size(2), D = kh->size(3);
    if (k->size(1) != H || k->size(2) != D || k->scalar_type() != at::kBFloat16 ||
        v->scalar_type() != at::kBFloat16 || k->stride(2) != 1 || v->stride(2) != 1 || !on(k, dev) || !on(v, dev) ||
        !is_index(pos, dev, at::kLong, B) || !is_index(slots, dev, at::kLong, B) ||
        !is_index(next, dev, at::kLong, B) || (!slots && B > N))
        Py_RETURN_FALSE;
    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ommx_ring_write(data<uint16_t>(k), data<uint16_t>(v), k->stride(0), k->stride(1), v->stride(0), v->stride(1),
                         data<uint16_t>(kh), data<uint16_t>(vh), kh->stride(0), rows, data<int64_t>(slots),
                         data<int64_t>(pos), data<int64_t>(next), B, H, D, sink, span, data<int32_t>(err), stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "ommx_ring_write")) return nullptr;
    Py_RETURN_TRUE;
}

// (k_hist, v_hist, k_tail, v_tail, span, seq, tail_idx, slots, b_tail_len, b_seq_len, window_sink, window_recent,
//  group_tokens, packed_lag, err_flag)
PyObject* py_tail_gather(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 15) { PyErr_SetString(PyExc_TypeError, "tail_gather: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *kh = as_tensor(a[0], ok), *vh = as_tensor(a[1], ok), *kt = as_tensor(a[2], ok),
                     *vt = as_tensor(a[3], ok), *seq = as_tensor_or_none(a[5], ok),
                     *idx = as_tensor_or_none(a[6], ok), *slots = as_tensor_or_none(a[7], ok),
                     *bt = as_tensor_or_none(a[8], ok), *bs = as_tensor_or_none(a[9], ok),
                     *err = as_tensor_or_none(a[14], ok);
    const int64_t span = as_int(a[4], ok), wsink = as_int(a[10], ok), recent = as_int(a[11], ok),
                  gt = as_int(a[12], ok), lag = as_int(a[13], ok);
    if (!ok || !is_history(*kh, *vh) || kt->dim() != 4 || kt->sizes() != vt->sizes() || !seq == !idx) Py_RETURN_FALSE;
    const c10::Device dev = kh->device();
    const int64_t B = kt->size(0), T = kt->size(1), N = kh->size(0), rows = kh->size(1), H = kh->size(2), D = kh->size(3);
    if (kt->size(2) != H || kt->size(3) != D || kt->scalar_type() != at::kBFloat16 ||
        vt->scalar_type() != at::kBFloat16 || !kt->is_contiguous() || !vt->is_contiguous() ||
        !is_index(seq, dev, at::kLong, B) || !is_index(idx, dev, at::kLong, B * T) ||
        !is_index(slots, dev, at::kLong, B) || !is_index(bt, dev, at::kInt, B) || !is_index(bs, dev, at::kInt, B) ||
        (!slots && B > N))
        Py_RETURN_FALSE;
    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ommx_tail_gather(data<uint16_t>(kh), data<uint16_t>(vh), kh->stride(0), rows, data<int64_t>(slots),
                          data<int64_t>(seq), data<int64_t>(idx), data<uint16_t>(kt), data<uint16_t>(vt),
                          data<int32_t>(bt), data<int32_t>(bs), B, T, H, D, wsink, recent, gt, span, lag,
                          data<int32_t>(err), stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "ommx_tail_gather")) return nullptr;
    Py_RETURN_TRUE;
}

// (K, V, k_hist, v_hist, request, pos0, n_head, lo, sink, span): rows [0, n_head) and [lo, T) of a block into the
// history of one request
PyObject* py_rows_write(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 10) { PyErr_SetString(PyExc_TypeError, "rows_write: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *K = as_tensor(a[0], ok), *V = as_tensor(a[1], ok), *kh = as_tensor(a[2], ok), *vh = as_tensor(a[3], ok);
    const int64_t pos0 = as_int(a[5], ok);
    PyObject* const rest[] = {a[2], a[3], a[4], a[6], a[7], a[8], a[9]};
    ommx::BlockRows rows;
    if (!ok) Py_RETURN_FALSE;
    at::Tensor copies[2];
    if (K->is_alias_of(*kh) || K->is_alias_of(*vh) || V->is_alias_of(*kh) || V->is_alias_of(*vh)) {
        // rows of the history itself: a launch writes them in no order
        copies[0] = K->clone();
        copies[1] = V->clone();
        K = &copies[0];
        V = &copies[1];
    }
    if (!read_block_rows(*K, *V, rest, pos0, rows)) Py_RETURN_FALSE;
    c10::hip::HIPGuard guard(K->device().index());
    hipStream_t stream = stream_of(K->device());
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ommx::rows_write(rows, stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "rows_write")) return nullptr;
    Py_RETURN_TRUE;
}

bool read_ints(PyObject* list, std::vector<int64_t>& out) {
    if (!PyList_Check(list)) return false;
    bool ok = true;
    const Py_ssize_t n = PyList_GET_SIZE(list);
    out.reserve(n);
    for (Py_ssize_t i = 0; i < n; ++i) out.push_back(as_int(PyList_GET_ITEM(list, i), ok));
    return ok;
}

// (k_hist, v_hist, planes, pairs [r0, g0, r1, g1, ...], page_size, hist sink, hist span, window_sink, groups_per_seq,
//  err_flag, table, recipe x 8): packs group g of request r for every pair, the rows read in place from the history
PyObject* py_pack_groups(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 19) { PyErr_SetString(PyExc_TypeError, "pack_groups: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *kh = as_tensor(a[0], ok), *vh = as_tensor(a[1], ok), *err = as_tensor_or_none(a[9], ok),
                     *table = as_tensor(a[10], ok);
    const int64_t ps = as_int(a[4], ok), sink = as_int(a[5], ok), span = as_int(a[6], ok), wsink = as_int(a[7], ok),
                  per_seq = as_int(a[8], ok);
    Recipe r;
    Planes p;
    std::vector<int64_t> pairs64;
    if (!ok || !is_history(*kh, *vh) || !read_recipe(a + 11, r) || !read_planes(a[2], r, p) || ps < 1 || r.gt % ps ||
        !read_ints(a[3], pairs64) || pairs64.empty() || pairs64.size() % 2)
        Py_RETURN_FALSE;
    const int64_t count = static_cast<int64_t>(pairs64.size()) / 2, ppg = r.gt / ps, N = kh->size(0), rows = kh->size(1);
    for (int64_t i = 0; i < count; ++i) {
        const int64_t req = pairs64[2 * i], g = pairs64[2 * i + 1];
        if (req < 0 || req >= N || g < 0 || g >= per_seq || (span == 0 && wsink + (g + 1) * r.gt > rows)) Py_RETURN_FALSE;
    }
    if (span > 0 && sink + span > rows) Py_RETURN_FALSE;
    const std::vector<int32_t> pairs(pairs64.begin(), pairs64.end());
    const c10::Device dev = kh->device();
    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = launch_ring_groups(*kh, *vh, pairs64, p, r, ps, sink, span, wsink, per_seq, *table, data<int32_t>(err), nullptr, stream);
    Py_END_ALLOW_THREADS
    if (rc != 1) {
        if (failed(rc, "ommx_store_pack")) return nullptr;
        Py_RETURN_TRUE;
    }
    const at::Tensor K = kh->view({N * rows, kh->size(2), kh->size(3)}), V = vh->view({N * rows, kh->size(2), kh->size(3)});
    // index tables: stream-ordered scratch, given back to torch's allocator when this call returns
    c10::DataPtr scratch = c10::GetAllocator(c10::DeviceType::CUDA)->allocate(count * (r.gt + ppg + 1) * sizeof(int32_t));
    int32_t *src = static_cast<int32_t*>(scratch.get()), *pages = src + count * r.gt, *groups = pages + count * ppg;
    Py_BEGIN_ALLOW_THREADS
    rc = ommx::pack_list(pairs.data(), count, src, pages, groups, r.gt, ppg, rows, sink, span, wsink, per_seq,
                         per_seq * ppg, stream);
    if (rc == 0)
        rc = launch_store(K, V, 0, p, r, count * r.gt, ps, src, pages, groups, *table, data<int32_t>(err), {}, stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "ommx_store_pack")) return nullptr;
    Py_RETURN_TRUE;
}

// (k_hist, v_hist, planes, K, V, slots [B], starts [B + 1], groups [B], page_size, window_sink, groups_per_seq, err_flag,
//  table, recipe x 8): rows starts[i] .. starts[i + 1] of K / V are the whole prompt of a fresh request in slot slots[i] of a
// history without a ring: the rows are copied and the first groups[i] groups packed, two launches for all requests.
PyObject* py_pack_prompts(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 21) { PyErr_SetString(PyExc_TypeError, "pack_prompts: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *kh = as_tensor(a[0], ok), *vh = as_tensor(a[1], ok), *K = as_tensor(a[3], ok), *V = as_tensor(a[4], ok),
                     *err = as_tensor_or_none(a[11], ok), *table = as_tensor(a[12], ok);
    const int64_t ps = as_int(a[8], ok), wsink = as_int(a[9], ok), per_seq = as_int(a[10], ok);
    Recipe r;
    Planes p;
    std::vector<int64_t> slots, starts, groups;
    if (!ok || !is_history(*kh, *vh) || !read_recipe(a + 13, r) || !read_planes(a[2], r, p) || ps < 1 || r.gt % ps || wsink < 0 ||
        !read_ints(a[5], slots) || !read_ints(a[6], starts) || !read_ints(a[7], groups) || !is_rows(*K) || !is_rows(*V) ||
        K->scalar_type() != at::kBFloat16 || V->scalar_type() != at::kBFloat16 || K->sizes() != V->sizes() ||
        K->device() != kh->device() || V->device() != kh->device() || K->is_alias_of(*kh) || K->is_alias_of(*vh) ||
        V->is_alias_of(*kh) || V->is_alias_of(*vh))
        Py_RETURN_FALSE;
    const int64_t B = static_cast<int64_t>(slots.size()), N = kh->size(0), rows = kh->size(1), H = kh->size(2), D = kh->size(3);
    if (B < 1 || B > ommx::kPromptsPerLaunch || static_cast<int64_t>(starts.size()) != B + 1 ||
        static_cast<int64_t>(groups.size()) != B || starts[0] < 0 || starts.back() > K->size(0) || K->size(1) != H || K->size(2) != D)
        Py_RETURN_FALSE;
    std::vector<bool> taken(static_cast<size_t>(N), false);
    std::vector<ommx::PromptRow> prompts(static_cast<size_t>(B));
    int64_t total = 0;
    for (int64_t i = 0; i < B; ++i) {
        const int64_t len = starts[i + 1] - starts[i], slot = slots[i];
        if (len < 1 || len > rows || slot < 0 || slot >= N || taken[slot] || groups[i] < 0 || groups[i] > per_seq ||
            (groups[i] > 0 && wsink + groups[i] * r.gt > len))
            Py_RETURN_FALSE;
        taken[slot] = true;
        prompts[i] = {static_cast<int32_t>(starts[i]), static_cast<int32_t>(starts[i + 1]), static_cast<int32_t>(slot),
                      static_cast<int32_t>(total)};
        total += groups[i];
    }
    if (N * per_seq * (r.gt / ps) > INT32_MAX) Py_RETURN_FALSE;
    const c10::Device dev = kh->device();
    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    const int64_t T = total * r.gt;
    // index tables: stream-ordered scratch, given back to torch's allocator when this call returns
    c10::DataPtr scratch = c10::GetAllocator(c10::DeviceType::CUDA)->allocate((T + T / ps + total + 1) * sizeof(int32_t));
    int32_t *src = static_cast<int32_t*>(scratch.get()), *pages = src + T, *dst = pages + T / ps;
    const ommx::PromptBlocks blocks{data<uint16_t>(K), data<uint16_t>(V), K->stride(0), K->stride(1), V->stride(0), V->stride(1),
                                    data<uint16_t>(kh), data<uint16_t>(vh), kh->stride(0), static_cast<int>(H),
                                    static_cast<int>(D), static_cast<int>(wsink), static_cast<int>(r.gt),
                                    static_cast<int>(ps), static_cast<int>(per_seq)};
    int rc, rc2 = 0;
    Py_BEGIN_ALLOW_THREADS
    rc = ommx::prompt_blocks(blocks, prompts.data(), static_cast<int>(B), static_cast<int32_t>(total), src, pages, dst, stream);
    if (rc == 0 && total > 0) rc2 = launch_store(*K, *V, 0, p, r, T, ps, src, pages, dst, *table, data<int32_t>(err), {}, stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "prompt_blocks") || failed(rc2, "ommx_store_pack")) return nullptr;
    Py_RETURN_TRUE;
}

// (q, planes, k_hist, v_hist, slots, seq, b_seq_len, req_to_token, req_to_group, out, sm_scale, page_size, max_seq_len,
//  mean_seq_len, ring sink, ring span, window sink, window recent, plain kernel, err_flag, recipe x 8): decode over a
// pool's planes with the tail rows read in place from its history; out bf16 or fp32.  An observed call is refused.
PyObject* py_decode_pool(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 28) { PyErr_SetString(PyExc_TypeError, "decode_pool: wrong number of arguments"); return nullptr; }
    PyObject* const rows[] = {a[0], a[9]};
    if (!plain_call(rows, 2)) Py_RETURN_FALSE;
    bool ok = true;
    DecodeCall c;
    Recipe r;
    Planes p;
    // a cache of ranks keeps the bitmask beside them as what the kernels read
    PyObject* recipe[8];
    std::copy(a + 20, a + 28, recipe);
    if (is_word(recipe[3], "combinadic")) recipe[3] = g_bitmap;
    if (!read_recipe(recipe, r) || !read_planes(a[1], r, p)) Py_RETURN_FALSE;
    c.q = as_tensor(a[0], ok); c.k_tail = as_tensor(a[2], ok); c.v_tail = as_tensor(a[3], ok);
    c.hist_slots = as_tensor_or_none(a[4], ok); c.hist_seq = as_tensor(a[5], ok); c.seq = as_tensor(a[6], ok);
    c.rt = as_tensor(a[7], ok); c.rg = as_tensor(a[8], ok); c.o = as_tensor(a[9], ok);
    c.sm_scale = as_double(a[10], ok); c.ps = as_int(a[11], ok); c.max_seq = std::max<int64_t>(1, as_int(a[12], ok));
    if (a[13] != Py_None) c.mean = as_double(a[13], ok);
    c.ring_sink = as_int(a[14], ok); c.ring_span = as_int(a[15], ok); c.win_sink = as_int(a[16], ok);
    c.win_recent = as_int(a[17], ok); c.force = as_bool(a[18], ok); c.err = as_tensor_or_none(a[19], ok);
    if (!ok) Py_RETURN_FALSE;
    c.k_base = p.k_base; c.k_scale = p.k_scale; c.k_zp = p.k_zp; c.k_index = p.index; c.k_oval = p.oval;
    c.v_main = p.v_main; c.v_scale = p.v_scale; c.v_zp = p.v_zp; c.ms = p.ms; c.mc = p.mc;
    c.k = r.k; c.bitmap = r.bitmap; c.want_map = p.ms != nullptr; c.int8 = r.mode == OMMX_SCALE_POW2_INT8;
    return answer(run_decode(c));
}

// (q, k, v, out, starts, scale): causal attention of prompt rows, out fp32 or bf16.  An observed call is refused, and
// so is an output that lies in the inputs (the caller's way through rows of its own serves it).
PyObject* py_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 6) { PyErr_SetString(PyExc_TypeError, "prefill: wrong number of arguments"); return nullptr; }
    if (!plain_call(a, 4)) Py_RETURN_FALSE;
    bool ok = true;
    const at::Tensor *q = as_tensor(a[0], ok), *k = as_tensor(a[1], ok), *v = as_tensor(a[2], ok), *o = as_tensor(a[3], ok);
    std::vector<int64_t> starts;
    const double scale = as_double(a[5], ok);
    if (!ok || !read_ints(a[4], starts) || starts.size() < 2 || starts[0] < 0 || !q->is_cuda()) Py_RETURN_FALSE;
    for (size_t i = 1; i < starts.size(); ++i)
        if (starts[i] < starts[i - 1] || starts[i] - starts[i - 1] > ommx::kPrefillMaxRows) Py_RETURN_FALSE;
    for (const at::Tensor* t : {q, k, v, o})
        if (t->dim() != 3 || t->stride(2) != 1 || t->device() != q->device() || t->size(0) < starts.back()) Py_RETURN_FALSE;
    const int64_t Hq = q->size(1), Hkv = k->size(1), D = q->size(2);
    if (k->size(2) != D || v->size(2) != D || v->size(1) != Hkv || o->size(1) != Hq || o->size(2) != D ||
        (D != 64 && D != 128) || Hkv < 1 || Hq % Hkv || !(scale > 0) ||
        std::max(k->stride(0), v->stride(0)) >= ommx::kPrefillMaxStride)
        Py_RETURN_FALSE;
    for (const at::Tensor* t : {q, k, v, o}) {
        const bool is16 = t->scalar_type() == at::kBFloat16;
        if ((!is16 && (t != o || t->scalar_type() != at::kFloat)) || t->stride(0) % 8 || t->stride(1) % 8 ||
            (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15))
            Py_RETURN_FALSE;
    }
    // K and V are read by workgroups that end later; a workgroup reads its own rows of q before it writes them
    const bool in_place = o->data_ptr() == q->data_ptr() && o->scalar_type() == q->scalar_type() && o->strides() == q->strides();
    if (share_memory(*o, *k) || share_memory(*o, *v) || (!in_place && share_memory(*o, *q))) Py_RETURN_FALSE;
    if (starts.back() == starts[0]) Py_RETURN_TRUE;
    c10::hip::HIPGuard guard(q->device().index());
    hipStream_t stream = stream_of(q->device());
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ommx::prefill_attention(data<uint16_t>(q), q->stride(0), q->stride(1), data<uint16_t>(k), k->stride(0),
                                 k->stride(1), data<uint16_t>(v), v->stride(0), v->stride(1), data(o),
                                 o->scalar_type() == at::kBFloat16, o->stride(0), o->stride(1), starts.data(),
                                 static_cast<int>(starts.size()) - 1, Hq, Hkv, D, scale, stream);
    Py_END_ALLOW_THREADS
    if (failed(rc, "prefill_attention")) return nullptr;
    written(*o);
    Py_RETURN_TRUE;
}

// (starts, q heads, head_dim): the form of the kernel such prompts take, 0 to 2 in the order of ommx::PrefillForm.
PyObject* py_prefill_form(PyObject*, PyObject* const* a, Py_ssize_t n) {
    bool ok = n == 3;
    std::vector<int64_t> starts;
    if (!ok || !read_ints(a[0], starts) || starts.size() < 2) { PyErr_SetString(PyExc_TypeError, "prefill_form: starts, heads and head_dim expected"); return nullptr; }
    const int64_t Hq = as_int(a[1], ok), D = as_int(a[2], ok);
    if (!ok) { PyErr_SetString(PyExc_ValueError, "prefill_form: integers expected"); return nullptr; }
    return PyLong_FromLong(static_cast<long>(ommx::prefill_form(starts.data(), static_cast<int>(starts.size()) - 1, Hq, D)));
}

// (dst, values, n64 = all or none): a contiguous GPU tensor filled from a list of ints by a launch.  int64 and int32
// tensors take one entry per value; an int32 tensor with n64 given holds n64 int64 values first, then int32 ones.
PyObject* py_upload(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 2 && n != 3) { PyErr_SetString(PyExc_TypeError, "upload: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor* dst = as_tensor(a[0], ok);
    std::vector<int64_t> values;
    if (!ok || !dst->is_cuda() || !dst->is_contiguous() || !read_ints(a[1], values)) Py_RETURN_FALSE;
    const int64_t count = static_cast<int64_t>(values.size());
    const bool wide = dst->scalar_type() == at::kLong;
    if (!wide && dst->scalar_type() != at::kInt) Py_RETURN_FALSE;
    const int64_t n64 = n == 3 ? as_int(a[2], ok) : (wide ? count : 0);
    if (!ok || n64 < 0 || n64 > count || (wide && n64 != count) || dst->numel() * (wide ? 2 : 1) != count + n64)
        Py_RETURN_FALSE;
    std::vector<int32_t> words(static_cast<size_t>(count + n64));
    std::memcpy(words.data(), values.data(), static_cast<size_t>(n64) * 8);
    std::copy(values.begin() + n64, values.end(), words.begin() + 2 * n64);
    c10::hip::HIPGuard guard(dst->device().index());
    const int rc = ommx::upload_words(static_cast<int32_t*>(dst->data_ptr()), words.data(),
                                      static_cast<int>(words.size()), stream_of(dst->device()));
    if (failed(rc, "upload")) return nullptr;
    Py_RETURN_TRUE;
}

// (block, length, boundary, sink rows, tail rows, packed length): the block of a one-request step (ommx::step_block)
PyObject* py_step_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 6) { PyErr_SetString(PyExc_TypeError, "step_block: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor* block = as_tensor(a[0], ok);
    const int64_t seq = as_int(a[1], ok), boundary = as_int(a[2], ok), sink = as_int(a[3], ok), tail = as_int(a[4], ok),
                  packed = as_int(a[5], ok);
    if (!ok || !block->is_cuda() || !block->is_contiguous() || block->scalar_type() != at::kInt || block->numel() < 6 ||
        block->numel() % 2 || reinterpret_cast<uintptr_t>(block->data_ptr()) % 8)
        Py_RETURN_FALSE;
    c10::hip::HIPGuard guard(block->device().index());
    if (failed(ommx::step_block(block->data_ptr<int32_t>(), static_cast<int>(block->numel() / 2 - 1), seq, boundary, sink, tail, packed,
                                stream_of(block->device())), "step_block"))
        return nullptr;
    Py_RETURN_TRUE;
}

// ── one step's host bookkeeping ────────────────────────────────────────────────────────────────
// A decode step of short contexts is some 20 us of GPU time a layer; the loops over its requests and the calls around its
// launches took longer than that in Python.  Plain lists of ints only: anything else is refused, and served by the
// caller's own loops.

// Whether slot slots[i] holds seqs[i] - behind tokens for all i: 1 yes, 0 no, -1 not plain lists.
int all_at(PyObject* seq_len, PyObject* slots, PyObject* seqs, int64_t behind) {
    if (!PyList_CheckExact(seq_len) || !PyList_CheckExact(slots) || !PyList_CheckExact(seqs) ||
        PyList_GET_SIZE(slots) != PyList_GET_SIZE(seqs))
        return -1;
    bool ok = true, all = true;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(slots); ++i) {
        const int64_t slot = as_int(PyList_GET_ITEM(slots, i), ok), seq = as_int(PyList_GET_ITEM(seqs, i), ok);
        if (!ok || slot < 0 || slot >= PyList_GET_SIZE(seq_len)) return -1;
        const int64_t held = as_int(PyList_GET_ITEM(seq_len, slot), ok);
        if (!ok) return -1;
        all = all && held == seq - behind;
    }
    return all;
}

// (seq_len, slots, seqs, behind)
PyObject* py_all_at(PyObject*, PyObject* const* a, Py_ssize_t n) {
    bool ok = n == 4;
    const int64_t behind = ok ? as_int(a[3], ok) : 0;
    const int r = ok ? all_at(a[0], a[1], a[2], behind) : -1;
    if (r < 0) Py_RETURN_NONE;
    return PyBool_FromLong(r);
}

// What one step does to a pool that is one token behind it.
struct StepRow { int64_t slot, len, done; };         // length after the step, packed groups before it
// False, with nothing done: not plain lists, a slot not one token behind, without room, or named twice.
bool read_step(PyObject* lens, PyObject* packed, PyObject* slots, PyObject* seqs, int64_t cap, std::vector<StepRow>& step) {
    if (all_at(lens, slots, seqs, 1) != 1 || !PyList_CheckExact(packed) || PyList_GET_SIZE(packed) != PyList_GET_SIZE(lens)) return false;
    const Py_ssize_t B = PyList_GET_SIZE(slots), N = PyList_GET_SIZE(lens);
    bool ok = true;
    step.resize(static_cast<size_t>(B));
    std::vector<bool> taken(static_cast<size_t>(N), false);
    for (Py_ssize_t i = 0; i < B; ++i) {
        StepRow& s = step[i];
        s.slot = as_int(PyList_GET_ITEM(slots, i), ok);
        s.len = as_int(PyList_GET_ITEM(lens, s.slot), ok) + 1;
        s.done = as_int(PyList_GET_ITEM(packed, s.slot), ok);
        if (!ok || s.len > cap || taken[s.slot]) return false;
        taken[s.slot] = true;
    }
    return true;
}
int64_t groups_after(const StepRow& s, int64_t kept, int64_t gt) { return s.len >= kept ? (s.len - kept) / gt : 0; }
// The pool's lengths moved; the list of (slot, first, end) of the groups that are complete with the step.
PyObject* finish_step(PyObject* lens, const std::vector<StepRow>& step, int64_t kept, int64_t gt) {
    PyObject* full = PyList_New(0);
    for (size_t i = 0; i < step.size() && full; ++i) {
        const StepRow& s = step[i];
        const int64_t target = groups_after(s, kept, gt);
        PyObject* item = nullptr;
        bool put = PyList_SetItem(lens, s.slot, PyLong_FromLongLong(s.len)) == 0;
        if (put && target > s.done) {
            item = Py_BuildValue("(LLL)", static_cast<long long>(s.slot), static_cast<long long>(s.done), static_cast<long long>(target));
            put = item && PyList_Append(full, item) == 0;
        }
        Py_XDECREF(item);
        if (!put) Py_CLEAR(full);
    }
    return full;
}

// (the arguments of ring_write without pos_next) + (seq_len, packed_groups, slots, seqs, kept rows, group_tokens, capacity or
// None): one row of every request of a step appended to a pool that is one token behind it.  Returns the list of
// (slot, first, end) of the groups that are complete with it (packed_groups is the caller's to move, once they are
// packed), or None with nothing done.
PyObject* py_append_rows(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    if (n != 16) { PyErr_SetString(PyExc_TypeError, "append_rows: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const int64_t kept = as_int(a[13], ok), gt = as_int(a[14], ok), cap = a[15] == Py_None ? INT32_MAX : as_int(a[15], ok);
    std::vector<StepRow> step;
    if (!ok || gt < 1 || !read_step(a[9], a[10], a[11], a[12], cap, step)) Py_RETURN_NONE;
    const at::Tensor* k = as_tensor(a[3], ok);
    if (!ok || k->dim() != 3 || k->size(0) != static_cast<int64_t>(step.size())) Py_RETURN_NONE;
    PyObject* const ring[] = {a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], Py_None, a[8]};
    PyObject* launched = py_ring_write(self, ring, 10);
    if (!launched) return nullptr;
    const bool done = launched == Py_True;
    Py_DECREF(launched);
    if (!done) Py_RETURN_NONE;
    return finish_step(a[9], step, kept, gt);
}

// (k_hist, v_hist, K, V, sink, span, err_flag, seq_len, packed_groups, slots, seqs, kept rows, group_tokens, capacity or None,
// block or None, store): append_rows of up to kStepRows requests with slots and positions as arguments of the launch, which also
// fills the int32 tensor block[7 B] (ommx::ring_step).  `store`: what pack_groups takes for this pool, (planes, page_size, window_sink,
// groups_per_seq, table, recipe x 8); the groups that are complete with the step are packed by the same launch, where that takes both.
// Returns (groups as append_rows, largest packed length, their sum, whether the groups are packed), or None with nothing done.
PyObject* py_append_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 16) { PyErr_SetString(PyExc_TypeError, "append_step: wrong number of arguments"); return nullptr; }
    bool ok = true;
    const at::Tensor *kh = as_tensor(a[0], ok), *vh = as_tensor(a[1], ok), *k = as_tensor(a[2], ok), *v = as_tensor(a[3], ok),
                     *err = as_tensor_or_none(a[6], ok), *block = as_tensor_or_none(a[14], ok);
    const int64_t sink = as_int(a[4], ok), span = as_int(a[5], ok), kept = as_int(a[11], ok), gt = as_int(a[12], ok),
                  cap = a[13] == Py_None ? INT32_MAX : as_int(a[13], ok);
    std::vector<StepRow> step;
    // (a larger batch is refused before its lists are read: the caller's other way reads them)
    if (!ok || gt < 1 || !PyList_CheckExact(a[9]) || PyList_GET_SIZE(a[9]) > ommx::kStepRows ||
        !read_step(a[7], a[8], a[9], a[10], std::min<int64_t>(cap, INT32_MAX), step))
        Py_RETURN_NONE;
    const int64_t B = static_cast<int64_t>(step.size());
    if (B < 1 || !is_history(*kh, *vh) || k->dim() != 3 || k->sizes() != v->sizes()) Py_RETURN_NONE;
    const c10::Device dev = kh->device();
    const int64_t N = kh->size(0), rows = kh->size(1), H = kh->size(2), D = kh->size(3);
    if (k->size(0) != B || k->size(1) != H || k->size(2) != D || k->scalar_type() != at::kBFloat16 ||
        v->scalar_type() != at::kBFloat16 || k->stride(2) != 1 || v->stride(2) != 1 || !on(k, dev) || !on(v, dev) ||
        !is_index(block, dev, at::kInt, 7 * B) || (block && reinterpret_cast<uintptr_t>(block->data_ptr()) % 8))
        Py_RETURN_NONE;
    ommx::StepWrite write;
    ommx::StepRows& at_rows = write.at;
    std::vector<int64_t> pairs;
    int64_t longest = 0, sum = 0;
    for (int64_t i = 0; i < B; ++i) {
        const StepRow& s = step[i];
        if (s.slot >= N) Py_RETURN_NONE;
        const int64_t packed = groups_after(s, kept, gt) * gt;
        at_rows.slot[i] = static_cast<int32_t>(s.slot);
        at_rows.pos[i] = static_cast<int32_t>(s.len - 1);
        at_rows.packed[i] = static_cast<int32_t>(packed);
        longest = std::max(longest, packed);
        sum += packed;
        for (int64_t g = s.done; g < packed / gt; ++g) { pairs.push_back(s.slot); pairs.push_back(g); }
    }
    c10::hip::HIPGuard guard(dev.index());
    hipStream_t stream = stream_of(dev);
    int rc = 1;
    bool together = false;
    if (!pairs.empty() && PyTuple_CheckExact(a[15]) && PyTuple_GET_SIZE(a[15]) == 13) {
        PyObject* how[13];
        for (int i = 0; i < 13; ++i) how[i] = PyTuple_GET_ITEM(a[15], i);
        Recipe r;
        Planes p;
        const int64_t ps = as_int(how[1], ok), wsink = as_int(how[2], ok), per_seq = as_int(how[3], ok);
        const at::Tensor* table = as_tensor(how[4], ok);
        auto rows16 = [](const at::Tensor* t) {
            return reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0 && t->stride(0) % 8 == 0 && t->stride(1) % 8 == 0;
        };
        bool fits = ok && read_recipe(how + 5, r) && read_planes(how[0], r, p) && r.gt == gt && ps >= 1 && gt % ps == 0 && (span == 0 || sink + span <= rows) &&
                    rows16(k) && rows16(v) && rows16(kh) && rows16(vh) && !k->is_alias_of(*kh) && !k->is_alias_of(*vh) && !v->is_alias_of(*kh) && !v->is_alias_of(*vh);
        // The workgroups of one launch run in any order: no group may hold the step's own token (a window without recent rows), nor a row whose place in
        // the ring that token takes.
        for (int64_t i = 0; i < B && fits; ++i) {
            const int64_t pos = step[i].len - 1, first = wsink + step[i].done * gt, end = wsink + at_rows.packed[i];
            if (step[i].done * gt >= at_rows.packed[i]) continue;
            fits = step[i].done >= 0 && at_rows.packed[i] / gt <= per_seq && end <= pos && (span == 0 ? end <= rows : first + span > pos);
        }
        if (fits) {
            write.k = data<uint16_t>(k); write.v = data<uint16_t>(v);
            write.k_bs = k->stride(0); write.k_hs = k->stride(1); write.v_bs = v->stride(0); write.v_hs = v->stride(1);
            write.k_hist = data<uint16_t>(kh); write.v_hist = data<uint16_t>(vh);
            write.stride_req = kh->stride(0);
            write.block = data<int32_t>(block); write.err = data<int32_t>(err);
            write.B = static_cast<int>(B); write.H = static_cast<int>(H); write.rows = static_cast<int>(rows);
            write.sink = static_cast<int>(sink); write.span = static_cast<int>(span);
            Py_BEGIN_ALLOW_THREADS
            rc = launch_ring_groups(*kh, *vh, pairs, p, r, ps, sink, span, wsink, per_seq, *table, data<int32_t>(err), &write, stream);
            Py_END_ALLOW_THREADS
            if (rc != 1 && failed(rc, "append_step")) return nullptr;
            together = rc == 0;
        }
    }
    if (!together) {
        Py_BEGIN_ALLOW_THREADS
        rc = ommx::ring_step(data<uint16_t>(k), data<uint16_t>(v), k->stride(0), k->stride(1), v->stride(0), v->stride(1),
                             data<uint16_t>(kh), data<uint16_t>(vh), kh->stride(0), rows, B, H, D, sink, span, at_rows,
                             data<int32_t>(block), data<int32_t>(err), stream);
        Py_END_ALLOW_THREADS
        if (failed(rc, "append_step")) return nullptr;
    }
    PyObject* full = finish_step(a[7], step, kept, gt);
    if (!full) return nullptr;
    return Py_BuildValue("(NLLO)", full, static_cast<long long>(longest), static_cast<long long>(sum), together ? Py_True : Py_False);
}

// (table, B): column 0 of the first B rows of a 2-D table of int32 or int64 in host memory as a list; None for anything else.
PyObject* py_first_column(PyObject*, PyObject* const* a, Py_ssize_t n) {
    bool ok = n == 2;
    const at::Tensor* t = ok ? as_tensor(a[0], ok) : nullptr;
    const int64_t B = ok ? as_int(a[1], ok) : 0;
    if (!ok || t->dim() != 2 || !t->is_cpu() || t->size(0) < B || t->size(1) < 1 || B < 0 || !plain_call(a, 1) ||
        (t->scalar_type() != at::kInt && t->scalar_type() != at::kLong))
        Py_RETURN_NONE;
    PyObject* out = PyList_New(B);
    for (int64_t i = 0; i < B && out; ++i) {
        const int64_t at = i * t->stride(0);
        PyObject* x = PyLong_FromLongLong(t->scalar_type() == at::kInt ? t->data_ptr<int32_t>()[at] : t->data_ptr<int64_t>()[at]);
        if (!x) Py_CLEAR(out);
        else PyList_SET_ITEM(out, i, x);
    }
    return out;
}

// C++ exceptions (out of memory among them) become the Python exceptions torch raises for them.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    return F(self, a, n);
    END_HANDLE_TH_ERRORS
}

#define OMMX_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<py_##name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    OMMX_FAST(auto_num_kv_splits), OMMX_FAST(plain), OMMX_FAST(rows_fit),
    OMMX_FAST(decode), OMMX_FAST(decode_pool), OMMX_FAST(store_pack), OMMX_FAST(pack_block), OMMX_FAST(pack_whole_block), OMMX_FAST(block_errors), OMMX_FAST(pack_groups), OMMX_FAST(pack_prompts), OMMX_FAST(ring_write),
    OMMX_FAST(all_at), OMMX_FAST(append_rows), OMMX_FAST(append_step), OMMX_FAST(first_column),
    OMMX_FAST(tail_gather), OMMX_FAST(rows_write), OMMX_FAST(upload), OMMX_FAST(step_block), OMMX_FAST(prefill), OMMX_FAST(prefill_form),
    {nullptr, nullptr, 0, nullptr},
};
#undef OMMX_FAST
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ommx_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ommx_host(void) {
    const char* names[] = {"k_base", "k_scale", "k_zp", "k_fp4_mapscale", "k_fp4_mapcenter", "k_obmp",
                           "k_oidx", "k_oval", "v_main", "v_scale", "v_zp"};
    for (int i = 0; i < 11; ++i)
        if (!(g_names[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
    if (!(g_bitmap = PyUnicode_InternFromString("bitmap"))) return nullptr;
    for (int i = 0; i < kBlockKeyCount; ++i)
        if (!(g_block_keys[i] = PyUnicode_InternFromString(kBlockKeys[i]))) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddIntConstant(m, "STEP_ROWS", ommx::kStepRows) < 0) Py_CLEAR(m);
    return m;
}

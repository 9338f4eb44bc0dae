// Launch path of the eager calls (module mlora._host): checks the tensors of a call, collects their addresses and
// calls the C ABI of libmlora_hip.so on torch's current stream.
//
// Why it is native: an eager decode or prefill step is a few calls per layer, each checking up to fourteen tensors.
// In Python that took 6 to 22 us a call on top of the launches themselves (2.6 us each), more than the kernels of a
// small batch run.  Host time per call, launches included, in Python -> here: plan_decode 9.2 -> 4.5 us, bgmv over seven
// projections in two launches 19.4 -> 9.1 us (0.5 of it the allocation of its intermediate), sgmv_multi over seven (three
// launches) 34.5 -> 10.7 us.
// The reference's q, k and v calls of a layer, outputs included (deltas_ref and Lora_GPU._invoke): 21 -> 16 us, a step of four layers
// that the host bounds 86 -> 65 us (66 since results are kept for one thread, stream and capture).
// Nothing is kept from one call for the next: every tensor is checked and every slab looked up on every call.  A negative
// code of the C ABI is returned, and raised by the caller.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/Allocator.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/mlora.h"

namespace {

struct PyFail {};   // a Python exception is set

[[noreturn]] void raise(PyObject *type, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    PyErr_FormatV(type, fmt, ap);
    va_end(ap);
    throw PyFail();
}

// ---------------------------------------------------------------- arguments
const at::Tensor &tensor(PyObject *o)
{
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, "expected a tensor, got %.100s", Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}

struct Ref {        // an owned reference
    PyObject *o;
    explicit Ref(PyObject *p) : o(p) { if (!o) throw PyFail(); }
    ~Ref() { Py_DECREF(o); }
    Ref(const Ref &) = delete;
    Ref &operator=(const Ref &) = delete;
};

PyObject *s_page_tbl, *s_rank, *s_scaling, *s_work, *s_group, *s_perm, *s_seg_start, *s_seg_len, *s_seg_adapter,
    *s_chunk_start, *s_chunk_len, *s_chunk_adapter, *s_counters, *s_row_off, *s_tok_rank, *s_tok_scale, *s_T, *s_workspace,
    *s_n_slots, *s_max_pages, *s_page_rows, *s_n_pages, *s_max_rank, *s_tok_adapter, *s_dtype_code, *s_projections, *s_a_rows, *s_b_rows, *s_buf;

void *attr_ptr(PyObject *o, PyObject *name)          // data pointer of a tensor attribute, null for None
{
    Ref a(PyObject_GetAttr(o, name));
    return a.o == Py_None ? nullptr : tensor(a.o).data_ptr();
}

long long as_int(PyObject *o)
{
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyFail();
    return v;
}

bool is_true(PyObject *o)
{
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw PyFail();
    return v != 0;
}

long long attr_int(PyObject *o, PyObject *name)
{
    Ref a(PyObject_GetAttr(o, name));
    return as_int(a.o);
}

void need_device(const at::Tensor &t)
{
    if (!t.is_cuda()) raise(PyExc_ValueError, "mlora kernels take device tensors; got a CPU tensor");
}

void need_contiguous(const at::Tensor &t)
{
    if (!t.is_contiguous()) raise(PyExc_ValueError, "mlora kernels take contiguous tensors");
}

struct List {       // a list or tuple of the caller
    PyObject *o;
    explicit List(PyObject *seq) : o(PySequence_Fast(seq, "expected a sequence")) { if (!o) throw PyFail(); }
    ~List() { Py_DECREF(o); }
    Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(o); }
    const at::Tensor &operator[](Py_ssize_t i) const { return tensor(PySequence_Fast_GET_ITEM(o, i)); }
};

void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

// Other Python threads run while a launch is made (it waits when the device's queue is full).
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    Unlocked() = default;
    ~Unlocked() { PyEval_RestoreThread(state); }
    Unlocked(const Unlocked &) = delete;
    Unlocked &operator=(const Unlocked &) = delete;
};

template <typename F, typename... A>
int launch(F entry_point, A... args)                 // args are read before the lock goes
{
    const Unlocked u;
    return entry_point(args...);
}

// ---------------------------------------------------------------- a call over projections of one pool layer
struct Call {
    int n = 0, dtype = 0;
    at::ScalarType type = at::kHalf;
    void *y[MLORA_MAX_PROJ];
    const void *x[MLORA_MAX_PROJ], *a[MLORA_MAX_PROJ], *b[MLORA_MAX_PROJ];
    int32_t hin[MLORA_MAX_PROJ], hout[MLORA_MAX_PROJ];
};

// Address of a layer of the slab tensor [n_layers, rows, width] that `slabs` (a dict) holds for a projection.
const void *slab_of(PyObject *slabs, PyObject *name, int64_t layer)
{
    Ref o(PyObject_GetItem(slabs, name));
    const at::Tensor &t = tensor(o.o);
    const int64_t l = layer < 0 ? layer + t.size(0) : layer;
    if (l < 0 || l >= t.size(0)) raise(PyExc_IndexError, "layer %lld outside the pool's %lld layers", (long long)layer, (long long)t.size(0));
    return static_cast<const char *>(t.data_ptr()) + l * t.stride(0) * t.element_size();
}

// The call's widths, slabs, y and x, after every check of their placement, type and shape.
Call call_of(PyObject *pool, PyObject *projs, int64_t layer, const List &ys, const List &xs, int64_t T)
{
    Call c;
    const Ref names(PySequence_Fast(projs, "expected the projections' names"));
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(names.o);
    if (n < 1 || n > MLORA_MAX_PROJ || ys.size() != n || xs.size() != n)
        raise(PyExc_ValueError, "need 1..%d projections with one y and one x each", MLORA_MAX_PROJ);
    for (Py_ssize_t i = 0; i < n; i++) { need_device(ys[i]); need_device(xs[i]); }
    for (Py_ssize_t i = 0; i < n; i++) { need_contiguous(ys[i]); need_contiguous(xs[i]); }
    c.n = (int)n;
    c.dtype = (int)attr_int(pool, s_dtype_code);
    c.type = c.dtype == MLORA_F16 ? at::kHalf : at::kBFloat16;
    const Ref widths(PyObject_GetAttr(pool, s_projections)), a_rows(PyObject_GetAttr(pool, s_a_rows)), b_rows(PyObject_GetAttr(pool, s_b_rows));
    for (Py_ssize_t i = 0; i < n; i++) {
        PyObject *name = PySequence_Fast_GET_ITEM(names.o, i);
        const Ref w(PyObject_GetItem(widths.o, name)), hi(PySequence_GetItem(w.o, 0)), ho(PySequence_GetItem(w.o, 1));
        c.hin[i] = (int32_t)as_int(hi.o);
        c.hout[i] = (int32_t)as_int(ho.o);
        const at::Tensor &yt = ys[i], &xt = xs[i];
        if (yt.scalar_type() != c.type || xt.scalar_type() != c.type)
            raise(PyExc_TypeError, "x and y must have the pool dtype %s", c.type == at::kHalf ? "torch.float16" : "torch.bfloat16");
        if (xt.dim() != 2 || yt.dim() != 2 || xt.size(0) != T || xt.size(1) != c.hin[i] || yt.size(0) != T || yt.size(1) != c.hout[i])
            raise(PyExc_ValueError, "projection %S: expected x [%lld, %d] and y [%lld, %d]", name, (long long)T, (int)c.hin[i],
                  (long long)T, (int)c.hout[i]);
        c.y[i] = yt.data_ptr();
        c.x[i] = xt.data_ptr();
        c.a[i] = slab_of(a_rows.o, name, layer);
        c.b[i] = slab_of(b_rows.o, name, layer);
    }
    return c;
}

struct Tables {
    const int32_t *page_tbl, *rank;
    const float *scaling;
    int n_slots, max_pages, page_rows, max_rank;
    int64_t n_pages;
};

Tables tables(PyObject *pool)
{
    return {static_cast<const int32_t *>(attr_ptr(pool, s_page_tbl)), static_cast<const int32_t *>(attr_ptr(pool, s_rank)),
            static_cast<const float *>(attr_ptr(pool, s_scaling)), (int)attr_int(pool, s_n_slots), (int)attr_int(pool, s_max_pages),
            (int)attr_int(pool, s_page_rows), (int)attr_int(pool, s_max_rank), attr_int(pool, s_n_pages)};
}

// ---------------------------------------------------------------- decode
// A plan's buffer: data pointer (null for None), after a check that a launch on `like` may write `n` values of its type there.
void *buffer(PyObject *plan, PyObject *name, at::ScalarType type, int64_t n, const at::Tensor &like)
{
    Ref a(PyObject_GetAttr(plan, name));
    if (a.o == Py_None) return nullptr;
    const at::Tensor &t = tensor(a.o);
    if (t.numel() < n)
        raise(PyExc_ValueError, "the plan's %U holds %lld values, %lld needed: it was made for a smaller batch or pool", name,
              (long long)t.numel(), (long long)n);
    if (t.scalar_type() != type || !t.is_contiguous() || t.device() != like.device())
        raise(PyExc_ValueError, "the plan's %U must be a contiguous buffer of its type on the batch's device", name);
    return t.data_ptr();
}

// gather(pool, plan, tok_adapter, group)
PyObject *gather(PyObject *const *v, Py_ssize_t nargs)
{
    if (nargs != 4) raise(PyExc_TypeError, "gather takes 4 arguments");
    PyObject *pool = v[0], *plan = v[1];
    const at::Tensor &tok = tensor(v[2]);
    const Tables tb = tables(pool);
    const int64_t T = tok.numel(), segs = T < tb.n_slots ? T : tb.n_slots;
    auto i32 = [&](PyObject *name, int64_t n) { return static_cast<int32_t *>(buffer(plan, name, at::kInt, n, tok)); };
    // the per-token view, which is None unless the caller asked for it
    int32_t *row_off = i32(s_row_off, T * tb.max_pages), *tok_rank = i32(s_tok_rank, T);
    float *tok_scale = static_cast<float *>(buffer(plan, s_tok_scale, at::kFloat, T, tok));
    int32_t *perm = i32(s_perm, T), *seg_start = i32(s_seg_start, segs), *seg_len = i32(s_seg_len, segs), *seg_adapter = i32(s_seg_adapter, segs);
    int32_t *chunk_start = i32(s_chunk_start, T), *chunk_len = i32(s_chunk_len, T), *chunk_adapter = i32(s_chunk_adapter, T);
    int32_t *counters = i32(s_counters, MLORA_CNT_WORDS), *work = i32(s_work, (int64_t)MLORA_WORK_CAP(T) * MLORA_WORK_WORDS);
    need_device(tok);
    const int rc = launch(mlora_pool_gather, static_cast<const int32_t *>(tok.data_ptr()), (int)T, tb.page_tbl, tb.rank, tb.scaling, tb.n_slots,
                          tb.max_pages, tb.page_rows, tb.n_pages, row_off, tok_rank, tok_scale, perm, seg_start, seg_len, seg_adapter,
                          chunk_start, chunk_len, chunk_adapter, (int)as_int(v[3]), counters, work, stream());
    return PyLong_FromLong(rc);
}

// bgmv(pool, layer, projs, ys, xs, tok_adapter, plan or None, fused: True, False or None (by the sizes), accumulate)
PyObject *bgmv(PyObject *const *v, Py_ssize_t nargs)
{
    if (nargs != 9) raise(PyExc_TypeError, "bgmv takes 9 arguments");
    PyObject *pool = v[0], *plan = v[6] == Py_None ? nullptr : v[6];
    const List ys(v[3]), xs(v[4]);
    const at::Tensor &tok = tensor(v[5]);
    const bool accumulate = v[8] == Py_True;
    bool fused = v[7] != Py_None && is_true(v[7]);
    need_device(tok);
    need_contiguous(tok);
    if (tok.scalar_type() != at::kInt) raise(PyExc_TypeError, "tok_adapter must be int32");
    const int64_t T = tok.numel();
    const Call c = call_of(pool, v[2], as_int(v[1]), ys, xs, T);
    if (plan) {
        Ref made_for(PyObject_GetAttr(plan, s_tok_adapter));
        if (tensor(made_for.o).numel() != T) raise(PyExc_ValueError, "plan was built for a different batch size");
    } else if (v[7] == Py_None) {
        fused = true;
    } else if (!fused) {
        raise(PyExc_ValueError, "the two-launch form needs a plan");
    }
    const Tables tb = tables(pool);
    const int group = plan ? (int)attr_int(plan, s_group) : 1;
    // The intermediate of the two-launch forms is this call's own, from torch's allocator: calls that share a plan may
    // overlap on several streams or threads, and a captured graph keeps what its launches write.  It may be given back
    // when the launches are queued (the allocator hands it out again in stream order).
    at::Tensor room;
    int64_t ws_bytes = 0;
    int form = MLORA_FORM_FUSED;
    if (!fused && T > 0) {
        form = mlora_bgmv_form(c.n, c.hin, c.hout, (int)T, tb.n_slots, tb.max_rank, group, &ws_bytes);
        if (form < 0) return PyLong_FromLong(form);
        if (v[7] != Py_None) form = MLORA_FORM_PAIR;
        if (form != MLORA_FORM_FUSED) room = at::empty({ws_bytes}, tok.options().dtype(at::kByte));
    }
    const int rc = launch(
        mlora_bgmv_multi_form, form, c.n, c.y, c.x, c.a, c.b, c.hin, c.hout, static_cast<const int32_t *>(tok.data_ptr()), (int)T, tb.page_tbl, tb.rank, tb.scaling,
        tb.n_slots, tb.max_pages, tb.page_rows, tb.n_pages, tb.max_rank, plan ? static_cast<const int32_t *>(attr_ptr(plan, s_work)) : nullptr,
        group, room.defined() ? room.data_ptr() : nullptr, ws_bytes, c.dtype, accumulate, stream());
    return PyLong_FromLong(rc);
}

// A reference-layout decode call over n projections: every check, then the launch.  y, x, a, b give the tensors of a projection.
template <typename Y, typename X, typename A, typename B>
int ref_call(PyObject *plan, int n, Y y_of, X x_of, A a_of, B b_of, int layer, float scale, bool accumulate, int64_t T, int64_t N, int64_t L, int64_t r)
{
    for (int i = 0; i < n; i++) { need_device(y_of(i)); need_device(x_of(i)); need_device(a_of(i)); need_device(b_of(i)); }
    for (int i = 0; i < n; i++) { need_contiguous(y_of(i)); need_contiguous(x_of(i)); need_contiguous(a_of(i)); need_contiguous(b_of(i)); }
    void *y[MLORA_MAX_PROJ];
    const void *x[MLORA_MAX_PROJ], *a[MLORA_MAX_PROJ], *b[MLORA_MAX_PROJ];
    int32_t hin[MLORA_MAX_PROJ], hout[MLORA_MAX_PROJ];
    const at::ScalarType type = y_of(0).scalar_type();
    int max_hin = 0;
    for (int i = 0; i < n; i++) {
        const at::Tensor &yt = y_of(i), &xt = x_of(i), &at = a_of(i), &bt = b_of(i);
        if (at.dim() != 4 || bt.dim() != 4) raise(PyExc_ValueError, "wa_T_all must be [N, L, r, Hin] and wb_T_all [N, L, Hout, r]");
        if (at.size(0) != N || at.size(1) != L || at.size(2) != r || bt.size(0) != N || bt.size(1) != L || bt.size(3) != r)
            raise(PyExc_ValueError, "pool tensors disagree with each other or with the plan on N, L or r");
        if (xt.dim() != 2 || yt.dim() != 2 || xt.size(0) != T || xt.size(1) != at.size(3) || yt.size(0) != T || yt.size(1) != bt.size(2))
            raise(PyExc_ValueError, "x must be [B, Hin] and y [B, Hout] for the plan's batch");
        if (yt.scalar_type() != type || xt.scalar_type() != type || at.scalar_type() != type || bt.scalar_type() != type)
            raise(PyExc_TypeError, "y, x and the pools must share one 16-bit dtype");
        y[i] = yt.data_ptr(); x[i] = xt.data_ptr(); a[i] = at.data_ptr(); b[i] = bt.data_ptr();
        hin[i] = (int32_t)at.size(3); hout[i] = (int32_t)bt.size(2);
        max_hin = hin[i] > max_hin ? hin[i] : max_hin;
    }
    if (type != at::kHalf && type != at::kBFloat16) raise(PyExc_TypeError, "mlora kernels take float16 or bfloat16 tensors");
    const int64_t bytes = mlora_bgmv_workspace_bytes(n, (int)T, max_hin, (int)r);
    // this call's own, as in bgmv; straight from torch's allocator, a tensor takes longer to make
    at::DataPtr room;
    if (bytes > 0) {
        const c10::DeviceGuard device(y_of(0).device());
        room = c10::GetAllocator(at::kCUDA)->allocate((size_t)bytes);
    }
    void *ws = room.get();
    return launch(mlora_bgmv_reflayout_multi, n, y, x, a, b, hin, hout, attr_ptr(plan, s_buf), (int)T, (int)N, (int)L, (int)r,
                  layer, scale, (int)attr_int(plan, s_group), type == at::kHalf ? MLORA_F16 : MLORA_BF16, accumulate, ws, bytes, stream());
}

// bgmv_ref(plan, ys, xs, was, wbs, layer, scale, accumulate, T, N, L, r)
PyObject *bgmv_ref(PyObject *const *v, Py_ssize_t nargs)
{
    if (nargs != 12) raise(PyExc_TypeError, "bgmv_ref takes 12 arguments");
    const List ys(v[1]), xs(v[2]), was(v[3]), wbs(v[4]);
    const int n = (int)ys.size();
    if (n < 1 || n > MLORA_MAX_PROJ || xs.size() != n || was.size() != n || wbs.size() != n)
        raise(PyExc_ValueError, "need 1..%d projections with one y, x, wa and wb each", MLORA_MAX_PROJ);
    return PyLong_FromLong(ref_call(v[0], n, [&](int i) -> const at::Tensor & { return ys[i]; }, [&](int i) -> const at::Tensor & { return xs[i]; },
                                    [&](int i) -> const at::Tensor & { return was[i]; }, [&](int i) -> const at::Tensor & { return wbs[i]; },
                                    (int)as_int(v[5]), (float)PyFloat_AsDouble(v[6]), v[7] == Py_True, as_int(v[8]), as_int(v[9]),
                                    as_int(v[10]), as_int(v[11])));
}

// deltas_ref(plan, x, weights (wa, wb of every projection in turn), layer, T, N, L, r): the deltas alone, in new tensors of x's
// type; a tuple of them, or the C ABI's negative code
PyObject *deltas_ref(PyObject *const *v, Py_ssize_t nargs)
{
    if (nargs != 8) raise(PyExc_TypeError, "deltas_ref takes 8 arguments");
    const at::Tensor &x = tensor(v[1]);
    const List w(v[2]);
    const int n = (int)w.size() / 2;
    if (n < 1 || n > MLORA_MAX_PROJ || w.size() != 2 * n) raise(PyExc_ValueError, "need 1..%d projections with one wa and wb each", MLORA_MAX_PROJ);
    need_device(x);
    at::Tensor y[MLORA_MAX_PROJ];
    for (int i = 0; i < n; i++) {
        if (w[2 * i + 1].dim() != 4) raise(PyExc_ValueError, "wa_T_all must be [N, L, r, Hin] and wb_T_all [N, L, Hout, r]");
        y[i] = at::empty({x.size(0), w[2 * i + 1].size(2)}, x.options());
    }
    const int rc = ref_call(v[0], n, [&](int i) -> const at::Tensor & { return y[i]; }, [&](int) -> const at::Tensor & { return x; },
                            [&](int i) -> const at::Tensor & { return w[2 * i]; }, [&](int i) -> const at::Tensor & { return w[2 * i + 1]; },
                            (int)as_int(v[3]), 1.0f, false, as_int(v[4]), as_int(v[5]), as_int(v[6]), as_int(v[7]));
    if (rc) return PyLong_FromLong(rc);
    Ref out(PyTuple_New(n));
    for (int i = 0; i < n; i++) {
        PyObject *t = THPVariable_Wrap(y[i]);
        if (!t) throw PyFail();
        PyTuple_SET_ITEM(out.o, i, t);
    }
    Py_INCREF(out.o);
    return out.o;
}

// What orders a program's work: thread, device, stream and capture number (0 outside a capture).  What is queued under equal values
// runs in the order it is queued.
struct Order {
    int64_t v[4];
    Order()
    {
        const c10::hip::HIPStream s = c10::hip::getCurrentHIPStream();
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        unsigned long long id = 0;
        // the null stream cannot be captured, and asking it during another stream's capture is an error
        if (s.stream() && hipStreamGetCaptureInfo(s.stream(), &status, &id) != hipSuccess)
            raise(PyExc_RuntimeError, "the capture state of the current stream is not known: %s", hipGetErrorString(hipGetLastError()));
        v[0] = (int64_t)PyThread_get_thread_ident();
        v[1] = s.device_index();
        v[2] = (int64_t)(uintptr_t)s.stream();
        v[3] = status == hipStreamCaptureStatusNone ? 0 : (int64_t)id;
    }
};

PyObject *bytes_of(const int64_t *v, Py_ssize_t n) { return PyBytes_FromStringAndSize(reinterpret_cast<const char *>(v), n * (Py_ssize_t)sizeof(int64_t)); }

// order(): it, as bytes to compare
PyObject *order(PyObject *const *, Py_ssize_t nargs)
{
    if (nargs != 0) raise(PyExc_TypeError, "order takes no arguments");
    const Order o;
    return bytes_of(o.v, 4);
}

// state(x, weights): the order, and which objects x and the weights are at which torch versions, as bytes to compare while the
// objects are alive.  One call for all of it: the q, k and v calls of a layer ask for it every time.
PyObject *state(PyObject *const *v, Py_ssize_t nargs)
{
    if (nargs != 2) raise(PyExc_TypeError, "state takes 2 arguments");
    const List w(v[1]);
    if (w.size() > 2 * MLORA_MAX_PROJ) raise(PyExc_ValueError, "at most %d weights", 2 * MLORA_MAX_PROJ);
    int64_t out[4 + 2 * (1 + 2 * MLORA_MAX_PROJ)];
    const Order o;
    for (int i = 0; i < 4; i++) out[i] = o.v[i];
    Py_ssize_t n = 4;
    auto add = [&](PyObject *t) { out[n++] = (int64_t)(uintptr_t)t; out[n++] = tensor(t)._version(); };
    add(v[0]);
    for (Py_ssize_t i = 0; i < w.size(); i++) add(PySequence_Fast_GET_ITEM(w.o, i));
    return bytes_of(out, n);
}

// ---------------------------------------------------------------- prefill
struct Segments { const int32_t *start, *len, *adapter; int64_t n; };

Segments segments(const at::Tensor &start, const at::Tensor &len, const at::Tensor &adapter)
{
    const at::Tensor *all[3] = {&start, &len, &adapter};
    for (const at::Tensor *t : all) need_device(*t);
    for (const at::Tensor *t : all) need_contiguous(*t);
    for (const at::Tensor *t : all)
        if (t->scalar_type() != at::kInt) raise(PyExc_TypeError, "segment arrays must be int32");
    const int64_t n = start.numel();
    if (len.numel() != n || adapter.numel() != n) raise(PyExc_ValueError, "seg_start, seg_len and seg_adapter must have the same length");
    return {static_cast<const int32_t *>(start.data_ptr()), static_cast<const int32_t *>(len.data_ptr()),
            static_cast<const int32_t *>(adapter.data_ptr()), n};
}

// prefill_plan(pool, seg_start, seg_len, seg_adapter, T, workspace, aligned)
PyObject *prefill_plan(PyObject *const *v, Py_ssize_t nargs)
{
    if (nargs != 7) raise(PyExc_TypeError, "prefill_plan takes 7 arguments");
    PyObject *pool = v[0];
    const Segments sg = segments(tensor(v[1]), tensor(v[2]), tensor(v[3]));
    const at::Tensor &ws = tensor(v[5]);
    need_device(ws);
    need_contiguous(ws);
    const Tables tb = tables(pool);
    const auto plan = v[6] == Py_True ? mlora_sgmv_plan_aligned : mlora_sgmv_plan;
    const int rc = launch(plan, sg.start, sg.len, sg.adapter, (int)sg.n, tb.page_tbl, tb.rank, tb.scaling, (int)as_int(v[4]),
                        tb.n_slots, tb.max_pages, tb.page_rows, tb.n_pages, tb.max_rank, ws.data_ptr(), ws.numel(), stream());
    return PyLong_FromLong(rc);
}

// sgmv_multi(pool, layer, projs, ys, xs, plan, accumulate)
PyObject *sgmv_multi(PyObject *const *v, Py_ssize_t nargs)
{
    if (nargs != 7) raise(PyExc_TypeError, "sgmv_multi takes 7 arguments");
    PyObject *pool = v[0], *plan = v[5];
    const List ys(v[3]), xs(v[4]);
    const int64_t T = attr_int(plan, s_T);
    const Call c = call_of(pool, v[2], as_int(v[1]), ys, xs, T);
    Ref start(PyObject_GetAttr(plan, s_seg_start)), len(PyObject_GetAttr(plan, s_seg_len)), adapter(PyObject_GetAttr(plan, s_seg_adapter)),
        wsp(PyObject_GetAttr(plan, s_workspace));
    const Segments sg = segments(tensor(start.o), tensor(len.o), tensor(adapter.o));
    const at::Tensor &ws = tensor(wsp.o);
    need_device(ws);
    need_contiguous(ws);
    const Tables tb = tables(pool);
    const int rc = launch(mlora_sgmv_multi_planned, c.n, c.y, c.x, c.a, c.b, c.hin, c.hout, sg.start, sg.len, sg.adapter, (int)sg.n, tb.page_tbl,
                                            tb.rank, tb.scaling, (int)T, tb.n_slots, tb.max_pages, tb.page_rows, tb.n_pages, tb.max_rank,
                                            c.dtype, v[6] == Py_True, ws.data_ptr(), ws.numel(), stream());
    return PyLong_FromLong(rc);
}

// ---------------------------------------------------------------- module
template <PyObject *(*F)(PyObject *const *, Py_ssize_t)>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    try {
        return F(args, nargs);
    } catch (const PyFail &) {
        return nullptr;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

#define MLORA_FN(name) {#name, (PyCFunction)(void (*)())entry<name>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MLORA_FN(gather), MLORA_FN(bgmv), MLORA_FN(bgmv_ref), MLORA_FN(deltas_ref), MLORA_FN(order), MLORA_FN(state), MLORA_FN(prefill_plan),
                         MLORA_FN(sgmv_multi), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Native launch path of mlora's eager calls.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host()
{
    const std::pair<PyObject **, const char *> names[] = {
        {&s_page_tbl, "page_tbl"}, {&s_rank, "rank"}, {&s_scaling, "scaling"}, {&s_work, "work"}, {&s_group, "group"},
        {&s_perm, "perm"}, {&s_seg_start, "seg_start"}, {&s_seg_len, "seg_len"}, {&s_seg_adapter, "seg_adapter"},
        {&s_chunk_start, "chunk_start"}, {&s_chunk_len, "chunk_len"}, {&s_chunk_adapter, "chunk_adapter"}, {&s_counters, "counters"},
        {&s_row_off, "row_off"}, {&s_tok_rank, "tok_rank"}, {&s_tok_scale, "tok_scale"}, {&s_T, "T"}, {&s_workspace, "workspace"},
        {&s_n_slots, "n_slots"}, {&s_max_pages, "max_pages"}, {&s_page_rows, "page_rows"}, {&s_n_pages, "n_pages"},
        {&s_max_rank, "max_rank"}, {&s_tok_adapter, "tok_adapter"}, {&s_dtype_code, "dtype_code"}, {&s_projections, "projections"},
        {&s_a_rows, "a_rows"}, {&s_b_rows, "b_rows"}, {&s_buf, "buf"}};
    for (const auto &p : names)
        if (!(*p.first = PyUnicode_InternFromString(p.second))) return nullptr;
    return PyModule_Create(&module);
}

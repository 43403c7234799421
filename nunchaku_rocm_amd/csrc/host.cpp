// Host side of an operator call in native code: the checks of the ordinary call and the argument block of the C entry.
//
// A launch of this library takes 5 to 20 us on the GPU for small problems; checking fifteen tensors and filling the block from
// Python took the host 12 to 20 us a call, and that was what such calls waited for (a linear of 512 tokens: 43 us a call, 22 of
// kernels).  Each function here looks at everything the Python operator would look at, writes the block and returns true (or
// the tensors it allocated for the call) -- or changes nothing and returns False as soon as anything is not the ordinary case:
// another device, a subclass, a tensor under a transform, a layout that needs a copy, an argument that is wrong.  The Python
// code of the operator then does the call or raises; it decides everything that is not the ordinary case, and nothing is
// remembered here from one call to the next.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cmath>
#include <cstring>
#include <string>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/Storage.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/svdq_mi355x.h"

namespace {

using at::Tensor;

PyObject *no() { Py_RETURN_FALSE; }

// A tensor as the kernels take it: exactly torch.Tensor or Parameter, on `device`, no more than its values in memory for the
// dispatcher (no subclass, transform or functionalization around it).  None leaves `t` undefined.
struct Reader {
    c10::DeviceIndex device = -1;
    bool ok = true;

    bool get(PyObject *o, Tensor &t, bool optional = false) {
        if (!ok) return false;
        if (o == Py_None) return ok = optional;
        if (Py_TYPE(o) != (PyTypeObject *)THPVariableClass && Py_TYPE(o) != (PyTypeObject *)ParameterClass) return ok = false;
        t = THPVariable_Unpack(o);
        const auto keys = t.key_set();
        if (!t.is_cuda() || t.layout() != at::kStrided || t.is_neg() || t.is_conj() ||
            keys.has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::Functionalize, c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::Batched})))
            return ok = false;
        if (device < 0) device = t.device().index();
        return ok = t.device().index() == device;
    }
    // every tensor fits, and its device is the current one
    bool done() const { return ok && device >= 0 && c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice().index() == device; }
};

template <typename Args>
struct Block {  // the ctypes structure to fill
    Py_buffer view{};
    bool ok;
    explicit Block(PyObject *o) { ok = PyObject_GetBuffer(o, &view, PyBUF_WRITABLE) == 0 && view.len == (Py_ssize_t)sizeof(Args); if (PyErr_Occurred()) PyErr_Clear(); }
    ~Block() { if (view.obj) PyBuffer_Release(&view); }
    Args &operator*() { return *(Args *)view.buf; }
};

const void *ptr(const Tensor &t) { return t.defined() ? t.const_data_ptr() : nullptr; }
bool al(const Tensor &t, uintptr_t n) { return ((uintptr_t)t.const_data_ptr() & (n - 1)) == 0; }
bool is16(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
bool bytes2d(const Tensor &t) { return t.dim() == 2 && t.element_size() == 1 && t.stride(1) == 1; }
bool fits(int64_t v) { return v >= 0 && v <= INT32_MAX; }
int code(at::ScalarType t) { return t == at::kBFloat16 ? SVDQ_BF16 : SVDQ_FP16; }
bool flag(PyObject *o, long &v) { v = PyLong_Check(o) ? PyLong_AsLong(o) : -1; return PyLong_Check(o) && !PyErr_Occurred(); }
// an allocation goes through torch.empty's Python surface when somebody listens there
bool listened() { return at::impl::PythonTorchFunctionTLS::stack_len() > 0; }

// An allocation may wait for the device, and with somebody else's allocator for another Python thread: not under the interpreter's lock.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
Tensor empty(at::IntArrayRef size, const at::Device &device, at::ScalarType type) {
    const Unlocked unlocked;
    return at::empty(size, at::TensorOptions().device(device).dtype(type));
}

// same_source((version, storage, place, shape, stride), tensor): _prep._same_source; None where it cannot tell
PyObject *same_source(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 2 || !PyTuple_Check(a[0]) || PyTuple_GET_SIZE(a[0]) != 5 || !THPStorage_Check(PyTuple_GET_ITEM(a[0], 1))) Py_RETURN_NONE;
    Reader r;
    Tensor t;
    if (!r.get(a[1], t) || t.is_inference()) Py_RETURN_NONE;
    PyObject *const *s = &PyTuple_GET_ITEM(a[0], 0);
    const auto &storage = THPStorage_Unpack(s[1]);
    PyObject *shape = s[3], *stride = s[4];
    if (!PyTuple_Check(shape) || !PyTuple_Check(stride)) Py_RETURN_NONE;
    bool same = PyLong_AsLongLong(s[0]) == (long long)t._version() &&
                (const char *)storage.data() + PyLong_AsLongLong(s[2]) == (const char *)t.const_data_ptr() &&
                PyTuple_GET_SIZE(shape) == t.dim() && PyTuple_GET_SIZE(stride) == t.dim();
    for (int64_t d = 0; same && d < t.dim(); d++)
        same = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d)) == t.size(d) && PyLong_AsLongLong(PyTuple_GET_ITEM(stride, d)) == t.stride(d);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    return PyBool_FromLong(same);
}

// quantize_buffers(input, rank, pad_size, out_blocked) -> (output, oscales, lora_act_out) of svdq_quantize_w4a4_act_fuse_lora_cuda
PyObject *quantize_buffers(PyObject *, PyObject *const *a, Py_ssize_t n) {
    long rank, pad, blocked;
    Reader r;
    Tensor x;
    if (n != 4 || listened() || !r.get(a[0], x) || !r.done() || x.dim() != 2 || !flag(a[1], rank) || !flag(a[2], pad) || !flag(a[3], blocked) || pad < 1 ||
        rank < 0 || x.size(1) % 64)
        return no();
    const int64_t rows = (x.size(0) + pad - 1) / pad * pad, k = x.size(1);
    const Tensor q = empty({rows, blocked >= 2 ? k * 3 / 4 : k / 2}, x.device(), at::kByte), s = empty({k / 64, rows}, x.device(), x.scalar_type()),
                 l = empty({rows, rank}, x.device(), at::kFloat);
    PyObject *out = PyTuple_New(3);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(q));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(s));
    PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(l));
    return out;
}

// quantize(args, input, output, oscales, lora_down, lora_down_t, lora_act_out, smooth, stats, scale, shift, norm_eps, out_blocked):
// no GLU or GELU, signed; norm_eps None: no norm, else one with one scale and shift for all rows
PyObject *quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 13) return no();
    Reader r;
    Tensor x, out, sc, down, downt, la, smooth, stats, scale, shift;
    long blocked;
    const bool norm = a[11] != Py_None;
    const float eps = !norm ? 0.0f : PyFloat_Check(a[11]) ? (float)PyFloat_AS_DOUBLE(a[11]) : -1.0f;  // (as the block holds it)
    if (!r.get(a[1], x) || !r.get(a[2], out) || !r.get(a[3], sc) || !r.get(a[4], down, true) || !r.get(a[5], downt, true) || !r.get(a[6], la, true) ||
        !r.get(a[7], smooth, true) || !r.get(a[8], stats, true) || !r.get(a[9], scale, true) || !r.get(a[10], shift, true) || !r.done() ||
        !flag(a[12], blocked) || blocked < 0 || blocked > 3 || eps < 0.0f)
        return no();
    if (x.dim() != 2 || !is16(x.scalar_type()) || x.stride(1) != 1 || x.stride(0) % 8 || !al(x, 16)) return no();
    const auto T = x.scalar_type();
    const int64_t M = x.size(0), K = x.size(1), kb = blocked >= 2 ? K * 3 / 4 : K / 2;
    if (K % 64 || !fits(M) || !fits(K) || !fits(x.stride(0))) return no();
    if (!bytes2d(out) || out.size(0) < M || !fits(out.stride(0))) return no();
    if (blocked && (!out.is_contiguous() || out.size(0) % 32 || out.size(1) != kb || !al(out, 16))) return no();
    if (sc.dim() != 2 || sc.scalar_type() != T || sc.stride(1) != 1 || sc.size(1) < M || sc.size(0) < K / 64 || !fits(sc.stride(0))) return no();
    if (blocked == 3 && (K % 512 || !sc.is_contiguous() || sc.size(0) != K / 64 || sc.size(1) != out.size(0) || !al(sc, 16))) return no();
    int64_t R = 0;
    if (down.defined()) {
        if (down.dim() != 2 || down.scalar_type() != T || down.size(0) != K) return no();
        R = down.size(1);
        if (R && (!downt.defined() || !la.defined() || la.dim() != 2 || la.scalar_type() != at::kFloat || la.stride(1) != 1 || la.size(0) < M || !fits(la.stride(0))))
            return no();
    }
    if (smooth.defined() && (smooth.scalar_type() != T || !smooth.is_contiguous() || smooth.numel() != K)) return no();
    int64_t stride = 1, batch = 0;
    if (norm) {
        if (!scale.defined() || !shift.defined() || scale.scalar_type() != T || shift.scalar_type() != T || scale.dim() < 1 || scale.dim() > 2 ||
            scale.dim() != shift.dim() || scale.numel() != K || shift.numel() != K || scale.size(-1) != K || shift.size(-1) != K)
            return no();
        stride = scale.stride(-1);
        batch = scale.dim() == 2 ? scale.stride(0) : K * stride;  // (one batch: not looked at)
        if (scale.strides() != shift.strides() || stride < 1 || !fits(stride) || !fits(batch) || (stats.defined() ? stats.scalar_type() != at::kFloat || stats.dim() != 2 || stats.size(0) != M ||
                                                                                                 stats.size(1) != 2 || !stats.is_contiguous() : !(eps > 0.0f)))
            return no();
    } else if (scale.defined() || shift.defined() || stats.defined()) {
        return no();
    }
    Block<svdq_quantize_args> b(a[0]);
    if (!b.ok) return no();
    svdq_quantize_args &q = *b;
    q = svdq_quantize_args{};
    q.x = ptr(x);
    q.smooth = ptr(smooth);
    q.lora_down_t = R ? ptr(downt) : nullptr;
    q.out = out.data_ptr();
    q.scales = sc.data_ptr();
    q.lora_act = R ? (float *)la.data_ptr() : nullptr;
    q.M = (int32_t)M, q.K = (int32_t)K, q.R = (int32_t)R;
    q.ld_x = (int32_t)x.stride(0), q.ld_out = (int32_t)out.stride(0), q.ld_scales = (int32_t)sc.stride(0), q.ld_lora_act = R ? (int32_t)la.stride(0) : 0;
    q.dtype = code(T);
    q.prologue = SVDQ_PRE_NONE;
    q.norm_stats = (const float *)ptr(stats);
    q.norm_scale = ptr(scale), q.norm_shift = ptr(shift);
    q.norm_ld = (int32_t)batch, q.norm_stride = (int32_t)stride;
    q.out_blocked = blocked >= 2 ? 2 : (int32_t)blocked, q.scales_blocked = blocked == 3;
    q.norm_eps = norm && !stats.defined() ? eps : 0.0f;
    Py_RETURN_TRUE;
}

// gemm(args, act, wgt, planes, out, qout, ascales, wscales, oscales, lora_act_in, lora_up, lora_down, lora_down_t, lora_down_blocked,
//      lora_act_out, norm_q, norm_k, rotary, rotary_blocked, bias, smooth, act_unsigned, fuse_swiglu, act_blocked, qout_blocked)
// -> True, or the scratch tensor the launch needs
PyObject *gemm(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 25) return no();
    Reader r;
    Tensor act, wgt, planes, out, qout, as, ws, os, la, up, down, downt, downb, lo, nq, nk, rot, rotb, bias, smooth;
    long uns, swiglu, ablk, qblk;
    if (!r.get(a[1], act) || !r.get(a[2], wgt) || !r.get(a[3], planes) || !r.get(a[4], out, true) || !r.get(a[5], qout, true) || !r.get(a[6], as) ||
        !r.get(a[7], ws) || !r.get(a[8], os, true) || !r.get(a[9], la, true) || !r.get(a[10], up, true) || !r.get(a[11], down, true) ||
        !r.get(a[12], downt, true) || !r.get(a[13], downb, true) || !r.get(a[14], lo, true) || !r.get(a[15], nq, true) || !r.get(a[16], nk, true) ||
        !r.get(a[17], rot, true) || !r.get(a[18], rotb, true) || !r.get(a[19], bias, true) || !r.get(a[20], smooth, true) || !r.done() ||
        !flag(a[21], uns) || !flag(a[22], swiglu) || !flag(a[23], ablk) || !flag(a[24], qblk) || ablk < 0 || ablk > 3 || qblk < 0 || qblk > 3)
        return no();
    const bool quant = qout.defined(), qk = rot.defined();
    if (quant != os.defined() || (quant && qk) || qk != nq.defined() || qk != nk.defined() || (!quant && !out.defined()) || (swiglu && (!quant || out.defined())) ||
        (quant ? down.defined() != lo.defined() : down.defined() || lo.defined()))
        return no();
    if (!bytes2d(act) || !bytes2d(wgt)) return no();
    const int64_t M = act.size(0), K = wgt.size(1) * 2, N = wgt.size(0), G = K / 64;
    if (act.size(1) != (ablk >= 2 ? K * 3 / 4 : K / 2) || K % 64 || !fits(M) || !fits(K) || !fits(N)) return no();
    const auto T = out.defined() ? out.scalar_type() : os.scalar_type();
    if (!is16(T)) return no();
    int64_t rows = M;
    if (out.defined()) {
        if (out.dim() != 2 || out.size(1) != N || out.stride(1) != 1 || out.size(0) > M || !fits(out.stride(0))) return no();
        rows = out.size(0);
    }
    for (const Tensor *s : {&as, &ws})
        if (s->dim() != 2 || s->scalar_type() != T || s->size(0) < G || s->size(1) < (s == &as ? M : N) || s->stride(1) != 1 || !fits(s->stride(0))) return no();
    if (bias.defined() && (bias.dim() != 1 || bias.scalar_type() != T || bias.size(0) < N || bias.stride(0) != 1)) return no();
    const int64_t R = la.defined() && up.defined() ? (up.dim() == 2 ? up.size(1) : -1) : 0;
    if (R < 0) return no();
    if (R && (la.dim() != 2 || la.scalar_type() != at::kFloat || up.scalar_type() != T || up.size(0) < N || la.size(0) < M || la.size(1) < R || la.stride(1) != 1 ||
              up.stride(1) != 1 || !fits(la.stride(0)) || !fits(up.stride(0))))
        return no();
    if (ablk && (!act.is_contiguous() || M % 32 || !al(act, 16))) return no();
    if (ablk == 3 && (K % 512 || !as.is_contiguous() || as.size(0) != G || as.size(1) != M || !al(as, 16))) return no();
    if (!fits(act.stride(0)) || !fits(wgt.stride(0))) return no();
    if (qk) {
        for (const Tensor *w : {&nq, &nk})
            if (w->scalar_type() != T || w->numel() != 128 || !w->is_contiguous()) return no();
        if (rot.scalar_type() != at::kFloat || !rot.is_contiguous() || rot.numel() != rows * 128 || !al(rot, 16) || !rotb.defined()) return no();
    }
    const int64_t NQ = swiglu ? N / 2 : N, R2 = quant && down.defined() ? (down.dim() == 2 ? down.size(1) : -1) : 0;
    if (quant) {
        if (N % 128 || M % 16 || (swiglu && N % 32) || R2 < 0) return no();
        if (!bytes2d(qout) || qout.size(0) < M || qout.size(1) != (qblk >= 2 ? NQ * 3 / 4 : NQ / 2) || !fits(qout.stride(0))) return no();
        if (os.dim() != 2 || os.scalar_type() != T || os.size(0) != NQ / 64 || os.size(1) < M || os.stride(1) != 1 || !fits(os.stride(0))) return no();
        if (smooth.defined() && (smooth.scalar_type() != T || smooth.numel() != NQ || !smooth.is_contiguous())) return no();
        if (R2 && (down.scalar_type() != T || down.size(0) != NQ || !downt.defined() || lo.dim() != 2 || lo.scalar_type() != at::kFloat || lo.size(0) < M ||
                   lo.size(1) != R2 || !fits(lo.stride(0)) || listened()))
            return no();
        if (qblk && (!qout.is_contiguous() || qout.size(0) % 32 || !al(qout, 16))) return no();
        if (qblk == 3 && (NQ % 512 || !os.is_contiguous() || os.size(1) != qout.size(0) || !al(os, 16))) return no();
    }
    Block<svdq_gemm_args> b(a[0]);
    if (!b.ok) return no();
    svdq_gemm_args &g = *b;
    g = svdq_gemm_args{};
    g.act = ptr(act), g.wgt = ptr(wgt), g.wgt_planes = ptr(planes), g.ascales = ptr(as), g.wscales = ptr(ws), g.bias = ptr(bias);
    g.lora_act = R ? (const float *)ptr(la) : nullptr, g.lora_up = R ? ptr(up) : nullptr;
    g.out = out.defined() ? out.data_ptr() : nullptr;
    g.M = (int32_t)M, g.N = (int32_t)N, g.K = (int32_t)K, g.R = (int32_t)R, g.actual_m = (int32_t)rows;
    g.ld_act = (int32_t)act.stride(0), g.ld_wgt = (int32_t)wgt.stride(0), g.ld_ascales = (int32_t)as.stride(0), g.ld_wscales = (int32_t)ws.stride(0);
    g.ld_lora_act = R ? (int32_t)la.stride(0) : 0, g.ld_lora_up = R ? (int32_t)up.stride(0) : 0, g.ld_out = out.defined() ? (int32_t)out.stride(0) : 0;
    g.dtype = code(T), g.act_unsigned = uns != 0;
    g.epilogue = qk ? SVDQ_EPI_QK_NORM_ROPE : !quant ? SVDQ_EPI_PLAIN : swiglu ? SVDQ_EPI_SWIGLU_QUANT : SVDQ_EPI_GELU_QUANT;
    g.eps = 1e-6f;
    g.act_blocked = ablk >= 2 ? 2 : (int32_t)ablk, g.ascales_blocked = ablk == 3;
    if (qk) {
        g.norm_q = ptr(nq), g.norm_k = ptr(nk), g.rotary = (const float *)ptr(rot), g.ld_rotary = 128, g.rotary_blocked = (const float *)ptr(rotb);
    }
    if (!quant) Py_RETURN_TRUE;
    g.qout = qout.data_ptr(), g.oscales = os.data_ptr(), g.smooth_next = ptr(smooth);
    g.R2 = (int32_t)R2, g.ld_qout = (int32_t)qout.stride(0), g.ld_oscales = (int32_t)os.stride(0);
    g.shift = swiglu ? 0.0f : 0.171875f;
    g.qout_blocked = qblk >= 2 ? 2 : (int32_t)qblk, g.oscales_blocked = qblk == 3;
    if (!R2) Py_RETURN_TRUE;
    g.lora_down_t = ptr(downt), g.lora_act_out = (float *)lo.data_ptr(), g.ld_lora_act_out = (int32_t)lo.stride(0);
    g.lora_down_blocked = ptr(downb);
    const Tensor scratch = empty({(N + SVDQ_LORA_PART_COLS - 1) / SVDQ_LORA_PART_COLS * M * R2}, act.device(), at::kFloat);
    g.scratch = (float *)scratch.data_ptr();
    return THPVariable_Wrap(scratch);
}

// gemv(args, x, kernel, scales, zeros, bias, m, n, k) -> (out, address of the bias or 0): one launch of the AWQ GEMV kernel
PyObject *gemv(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 9 || listened()) return no();
    Reader r;
    Tensor x, w, s, z, bias;
    long m, nn, k;
    if (!r.get(a[1], x) || !r.get(a[2], w) || !r.get(a[3], s) || !r.get(a[4], z) || !r.get(a[5], bias, true) || !r.done() || !flag(a[6], m) || !flag(a[7], nn) ||
        !flag(a[8], k) || m < 1 || m > 32 || nn < 1 || k < 1 || nn % 32)
        return no();
    const auto T = x.scalar_type();
    if (x.dim() != 2 || x.size(0) != m || x.size(1) != k || !is16(T) || x.stride(1) != 1 || x.stride(0) % 8 || !al(x, 16) || !fits(x.stride(0))) return no();
    if ((int64_t)w.element_size() * w.numel() != (int64_t)nn * k / 2 || !w.is_contiguous() || (int64_t)nn * k / 2 >= (int64_t)1 << 32) return no();
    if (s.dim() != 2 || z.dim() != 2 || s.stride(1) != 1 || z.strides() != s.strides() || s.scalar_type() != T || z.scalar_type() != T || !fits(s.stride(0))) return no();
    if (k % 64 || s.size(0) < k / 64 || s.size(1) < nn || z.sizes() != s.sizes()) return no();
    // a bias with a gradient or a tangent wanted through it is an addition of its own
    if (bias.defined() && ((bias.requires_grad() && at::GradMode::is_enabled()) || bias._fw_grad(0).defined() || bias.scalar_type() != T || bias.dim() != 1 ||
                           bias.size(0) != nn || !bias.is_contiguous()))
        return no();
    Block<svdq_awq_gemv_args> b(a[0]);
    if (!b.ok) return no();
    const Tensor out = empty({m, nn}, x.device(), T);
    *b = svdq_awq_gemv_args{ptr(x), (const int32_t *)ptr(w), ptr(s), ptr(z), out.data_ptr(), (int32_t)m, (int32_t)nn, (int32_t)k, (int32_t)x.stride(0),
                            (int32_t)s.stride(0), (int32_t)nn, code(T)};
    PyObject *res = PyTuple_New(2);
    if (!res) return nullptr;
    PyTuple_SET_ITEM(res, 0, THPVariable_Wrap(out));
    PyTuple_SET_ITEM(res, 1, PyLong_FromVoidPtr(bias.defined() ? (void *)bias.const_data_ptr() : nullptr));
    return res;
}

// attention(args, query, key, value) -> out (B, T, H D), for scaled_dot_product_attention's covered case
PyObject *attention(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 4 || listened()) return no();
    Reader r;
    Tensor t[3];
    for (int i = 0; i < 3; i++)
        if (!r.get(a[1 + i], t[i])) return no();
    const Tensor &q = t[0], &k = t[1], &v = t[2];
    if (!r.done() || q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || !is16(q.scalar_type())) return no();
    const int64_t B = q.size(0), H = q.size(1), Tq = q.size(2), D = q.size(3), Tk = k.size(2);
    if ((D != 128 && D != 64) || Tk < 1 || !fits(B) || !fits(H) || !fits(Tq) || !fits(Tk)) return no();
    for (int i = 0; i < 3; i++) {
        if (t[i].scalar_type() != q.scalar_type() || t[i].stride(3) != 1 || !al(t[i], 16)) return no();
        if (i && (t[i].size(0) != B || t[i].size(1) != H || t[i].size(2) != Tk || t[i].size(3) != D)) return no();
        for (int d = 0; d < 3; d++)
            if (t[i].stride(d) % 8) return no();
    }
    Block<svdq_attention_args> b(a[0]);
    if (!b.ok) return no();
    const Tensor out = empty({B, Tq, H * D}, q.device(), q.scalar_type());
    svdq_attention_args &g = *b;
    g = svdq_attention_args{};
    g.q = ptr(q), g.k = ptr(k), g.v = ptr(v), g.o = out.data_ptr();
    g.sqb = q.stride(0), g.sqh = q.stride(1), g.sqm = q.stride(2);
    g.skb = k.stride(0), g.skh = k.stride(1), g.skn = k.stride(2);
    g.svb = v.stride(0), g.svh = v.stride(1), g.svn = v.stride(2);
    g.sob = out.stride(0), g.som = out.stride(1);
    g.B = (int32_t)B, g.H = (int32_t)H, g.Tq = (int32_t)Tq, g.Tkv = (int32_t)Tk, g.D = (int32_t)D, g.dtype = code(q.scalar_type());
    g.scale = (float)std::pow((double)D, -0.5);
    return THPVariable_Wrap(out);
}

// A C++ exception (an allocation that failed, say) becomes the Python one torch would raise.
template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *self, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    return F(self, a, n);
    END_HANDLE_TH_ERRORS
}

#define SVDQ_METHOD(f) {#f, (PyCFunction)(void (*)(void))guarded<f>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {SVDQ_METHOD(same_source), SVDQ_METHOD(quantize_buffers), SVDQ_METHOD(quantize), SVDQ_METHOD(gemm), SVDQ_METHOD(gemv),
                         SVDQ_METHOD(attention), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The tensors' layout and the interpreter's are those of the headers this was compiled with: under others it does not load.
PyMODINIT_FUNC PyInit__host(void) {
    const std::string python = std::to_string(PY_MAJOR_VERSION) + "." + std::to_string(PY_MINOR_VERSION) + ".";
    if (std::strncmp(Py_GetVersion(), python.c_str(), python.size()) != 0)
        return PyErr_Format(PyExc_ImportError, "built for Python %s, this is %s", PY_VERSION, Py_GetVersion());
    PyObject *torch = PyImport_ImportModule("torch"), *version = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
    Py_XDECREF(torch);
    const char *text = version ? PyUnicode_AsUTF8(version) : nullptr;
    const bool same = text && std::strcmp(text, SVDQ_TORCH_VERSION) == 0;
    if (text && !same) PyErr_Format(PyExc_ImportError, "built for torch %s, this is %s", SVDQ_TORCH_VERSION, text);
    Py_XDECREF(version);
    if (!same) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (m) PyModule_AddIntConstant(m, "ABI_VERSION", SVDQ_ABI_VERSION);
    return m;
}

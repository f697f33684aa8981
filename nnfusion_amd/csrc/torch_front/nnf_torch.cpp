// The per-call path of nnfusion_amd/ops.py: torch tensors in, one call of the C ABI (include/nnf_hip_kernels.h) out.
//
// A decode step is a run of kernels of 4 - 11 us each; the same calls through ctypes (argument checks, sizes and pointers
// taken from the tensors one Python attribute at a time, a foreign call of up to twenty converted arguments) took the host
// 10 - 13 us apiece, so that a step of twelve calls was bound by the interpreter.  Here a call checks its tensors, allocates
// what the caller did not bring and enters the library in about a microsecond.  No state is kept between calls.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>

#include "nnf_hip_kernels.h"

namespace
{
    using at::Tensor;

    PyObject* g_error = nullptr; // nnfusion_amd.ops.NnfError(status, where)

    // thrown with the Python error set
    struct Raised
    {
    };
    [[noreturn]] void raise(PyObject* type, const char* text)
    {
        PyErr_SetString(type, text);
        throw Raised();
    }
    void require(bool ok, const char* text)
    {
        if (!ok)
            raise(PyExc_AssertionError, text);
    }
    // one call of the library, the interpreter released meanwhile (a launch into a full queue waits)
    template <typename F, typename... Args>
    void call(const char* where, F* function, Args... args)
    {
        PyThreadState* const thread = PyEval_SaveThread();
        const int status = function(args...);
        PyEval_RestoreThread(thread);
        if (status == NNF_OK)
            return;
        PyObject* const e = g_error ? PyObject_CallFunction(g_error, "is", status, where) : nullptr;
        if (e)
            PyErr_SetObject(g_error, e);
        Py_XDECREF(e);
        throw Raised();
    }

    const Tensor& tensor(PyObject* o)
    {
        if (!THPVariable_Check(o))
            raise(PyExc_TypeError, "a torch.Tensor is expected");
        return THPVariable_Unpack(o);
    }
    // the address of a tensor, or null for None
    void* address(PyObject* o) { return o == Py_None ? nullptr : tensor(o).data_ptr(); }
    int integer(PyObject* o)
    {
        const long v = PyLong_AsLong(o);
        if (v == -1 && PyErr_Occurred())
            throw Raised();
        if (v != (int)v)
            raise(PyExc_OverflowError, "integer argument out of range");
        return (int)v;
    }
    float real(PyObject* o)
    {
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred())
            throw Raised();
        return (float)v;
    }
    void matrix(const Tensor& t)
    {
        if (t.dim() != 2)
            raise(PyExc_ValueError, "a matrix is expected");
    }
    nnf_stream_t stream() { return (nnf_stream_t)c10::hip::getCurrentHIPStream().stream(); }

    // The caller's output buffer, or a new one.  `object`: what the Python caller gets back
    struct Output
    {
        PyObject* object = nullptr;
        void* data = nullptr;
        Output(PyObject* given, int m, int n, at::ScalarType type, const Tensor& like)
        {
            if (given != Py_None)
            {
                data = tensor(given).data_ptr();
                Py_INCREF(given);
                object = given;
                return;
            }
            Tensor t = at::empty({m, n}, like.options().dtype(type));
            data = t.data_ptr();
            object = THPVariable_Wrap(std::move(t));
            if (!object)
                throw Raised();
        }
        ~Output() { Py_XDECREF(object); }
        PyObject* release()
        {
            PyObject* o = object;
            object = nullptr;
            return o;
        }
    };
    // The caller's workspace, or one of `need()` bytes for this call (torch's allocator keeps the block for the next)
    struct Workspace
    {
        Tensor own;
        void* data = nullptr;
        size_t bytes = 0;
        template <typename F>
        Workspace(PyObject* given, const Tensor& like, F need)
        {
            if (given != Py_None)
            {
                const Tensor& t = tensor(given);
                data = t.data_ptr();
                bytes = (size_t)t.numel();
                return;
            }
            const size_t n = need();
            bytes = n > 16 ? n : 16;
            own = at::empty({(int64_t)bytes}, like.options().dtype(at::kByte));
            data = own.data_ptr();
        }
    };
    // nnf_plan with nothing but the synchronisation words, or a null pointer where the caller passed none
    struct SyncPlan
    {
        nnf_plan plan = {};
        const nnf_plan* ptr = nullptr;
        SyncPlan(PyObject* sync, int spin_limit = 0)
        {
            if (sync == Py_None)
                return;
            const Tensor& t = tensor(sync);
            plan.sync_flags = t.data_ptr();
            plan.sync_flags_bytes = (size_t)t.nbytes();
            plan.spin_limit = spin_limit;
            ptr = &plan;
        }
    };
    nnf_quant quant(PyObject* bits, PyObject* group, PyObject* zp, PyObject* zero_points)
    {
        return nnf_quant{integer(bits), integer(group), integer(zp), address(zero_points)};
    }

    using Args = PyObject* const*;

    // (a, wq, scales, group, zp, out, workspace)
    PyObject* w4a16_gemm(Args v)
    {
        const Tensor &a = tensor(v[0]), &wq = tensor(v[1]), &s = tensor(v[2]);
        matrix(a), matrix(wq), matrix(s);
        const int m = (int)a.size(0), k = (int)a.size(1), n = (int)wq.size(0), group = integer(v[3]);
        require(a.scalar_type() == at::kHalf && wq.scalar_type() == at::kByte && s.scalar_type() == at::kHalf, "fp16 activations, uint8 weights, fp16 scales");
        require(a.is_contiguous() && wq.is_contiguous() && s.is_contiguous(), "contiguous operands");
        require(group > 0 && wq.size(1) * 2 == k && s.size(0) == n && s.size(1) == k / group, "shapes of weights and scales");
        Output y(v[5], m, n, at::kHalf, a);
        Workspace w(v[6], a, [&] { return nnf_w4a16_gemm_workspace_bytes(m, n, k, group); });
        call("nnf_w4a16_gemm", nnf_w4a16_gemm, stream(), a.data_ptr(), wq.data_ptr(), s.data_ptr(), y.data, m, n, k, group, integer(v[4]),
             w.data, w.bytes);
        return y.release();
    }

    // (a, wq, scales, bits, group, zp, zero_points, out, workspace, sync, spin_limit)
    PyObject* wna16_gemm(Args v)
    {
        const Tensor &a = tensor(v[0]), &wq = tensor(v[1]), &s = tensor(v[2]);
        matrix(a), matrix(wq), matrix(s);
        const int m = (int)a.size(0), k = (int)a.size(1), n = (int)wq.size(0);
        const nnf_quant q = quant(v[3], v[4], v[5], v[6]);
        require(a.scalar_type() == at::kHalf && wq.scalar_type() == at::kByte && s.scalar_type() == at::kHalf, "fp16 activations, uint8 weights, fp16 scales");
        require(a.is_contiguous() && wq.is_contiguous() && s.is_contiguous(), "contiguous operands");
        require(q.group > 0 && wq.size(1) * 8 == (int64_t)k * q.bits && s.size(0) == n && s.size(1) == k / q.group, "shapes of weights and scales");
        if (q.zero_points)
        {
            const Tensor& z = tensor(v[6]);
            require(z.scalar_type() == at::kByte && z.is_contiguous(), "zero points: contiguous uint8");
            require(z.dim() == 2 && z.size(0) == n && z.size(1) == (k / q.group * q.bits + 7) / 8, "shape of the zero points");
        }
        Output y(v[7], m, n, at::kHalf, a);
        Workspace w(v[8], a, [&] { return nnf_wna16_gemm_preferred_workspace_bytes(m, n, k, &q); });
        const SyncPlan plan(v[9], integer(v[10]));
        call(plan.ptr ? "nnf_wna16_gemm_planned" : "nnf_wna16_gemm", nnf_wna16_gemm_planned, stream(), a.data_ptr(), wq.data_ptr(),
             s.data_ptr(), y.data, m, n, k, &q, plan.ptr, w.data, w.bytes);
        return y.release();
    }

    // (a, wq, scales, group, zp, rms_gamma, rms_eps, bias, residual, act, out, workspace, sync, spin_limit)
    PyObject* w4a16_gemm_fused(Args v)
    {
        const Tensor &a = tensor(v[0]), &wq = tensor(v[1]), &s = tensor(v[2]);
        matrix(a);
        const int m = (int)a.size(0), k = (int)a.size(1), group = integer(v[3]), zp = integer(v[4]), act = integer(v[9]);
        const int rows = (int)wq.size(0), n = rows / (act == NNF_ACT_SILU_GATE ? 2 : 1);
        Output y(v[10], m, n, at::kHalf, a);
        const SyncPlan plan(v[12], integer(v[13]));
        Workspace w(v[11], a, [&] {
            const size_t need = nnf_w4a16_gemm_fused_workspace_bytes(m, n, k, group, act);
            return plan.ptr ? need + nnf_w4a16_gemm_variant_workspace_bytes(m, rows, k, group, NNF_W4A16_AUTO, plan.ptr) : need;
        });
        call(plan.ptr ? "nnf_w4a16_gemm_fused_variant" : "nnf_w4a16_gemm_fused", nnf_w4a16_gemm_fused_variant, stream(), a.data_ptr(),
             wq.data_ptr(), s.data_ptr(), y.data, m, n, k, group, zp, address(v[5]), real(v[6]), address(v[7]), address(v[8]), act,
             NNF_W4A16_AUTO, plan.ptr, w.data, w.bytes);
        return y.release();
    }

    // (x, gamma, wgu, sgu, wd, sd, eps, group, zp, out, workspace, sync, spin_limit)
    PyObject* fused_mlp_w4a16(Args v)
    {
        const Tensor& x = tensor(v[0]);
        matrix(x);
        const int m = (int)x.size(0), h = (int)x.size(1), i = (int)(tensor(v[2]).size(0) / 2), group = integer(v[7]);
        Output y(v[9], m, h, at::kHalf, x);
        Workspace w(v[10], x, [&] { return nnf_fused_mlp_w4a16_workspace_bytes(m, h, i, group); });
        const SyncPlan plan(v[11], integer(v[12]));
        call(plan.ptr ? "nnf_fused_mlp_w4a16_planned" : "nnf_fused_mlp_w4a16", nnf_fused_mlp_w4a16_planned, stream(), x.data_ptr(),
             address(v[1]), real(v[6]), address(v[2]), address(v[3]), address(v[4]), address(v[5]), y.data, m, h, i, group, integer(v[8]),
             plan.ptr, plan.ptr, w.data, w.bytes);
        return y.release();
    }

    // (a, wq, scales, bits, group, zp, zero_points, rms_gamma, rms_eps, bias, residual, act, out, workspace)
    PyObject* wna16_gemm_fused(Args v)
    {
        const Tensor &a = tensor(v[0]), &wq = tensor(v[1]), &s = tensor(v[2]);
        matrix(a);
        const int m = (int)a.size(0), k = (int)a.size(1), act = integer(v[11]), n = (int)(wq.size(0) / (act == NNF_ACT_SILU_GATE ? 2 : 1));
        const nnf_quant q = quant(v[3], v[4], v[5], v[6]);
        Output y(v[12], m, n, at::kHalf, a);
        Workspace w(v[13], a, [&] { return nnf_wna16_gemm_fused_workspace_bytes(m, n, k, &q, act); });
        call("nnf_wna16_gemm_fused", nnf_wna16_gemm_fused, stream(), a.data_ptr(), wq.data_ptr(), s.data_ptr(), y.data, m, n, k, &q,
             address(v[7]), real(v[8]), address(v[9]), address(v[10]), act, w.data, w.bytes);
        return y.release();
    }

    // (x, gamma, wgu, sgu, wd, sd, bits, group, zp, zgu, zd, eps, out, workspace)
    PyObject* fused_mlp_wna16(Args v)
    {
        const Tensor& x = tensor(v[0]);
        matrix(x);
        const int m = (int)x.size(0), h = (int)x.size(1), i = (int)(tensor(v[2]).size(0) / 2);
        const nnf_quant qa = quant(v[6], v[7], v[8], v[9]), qb = quant(v[6], v[7], v[8], v[10]);
        Output y(v[12], m, h, at::kHalf, x);
        Workspace w(v[13], x, [&] { return nnf_fused_mlp_wna16_workspace_bytes(m, h, i, &qa, &qb); });
        call("nnf_fused_mlp_wna16", nnf_fused_mlp_wna16, stream(), x.data_ptr(), address(v[1]), real(v[11]), address(v[2]), address(v[3]),
             address(v[4]), address(v[5]), y.data, m, h, i, &qa, &qb, w.data, w.bytes);
        return y.release();
    }

    // the raw int32 accumulators (no scales) or the fp16 product
    PyObject* w8a8(const Tensor& a, const Tensor& b, const Tensor* s_tok, const Tensor* s_ch, PyObject* out, PyObject* workspace, PyObject* sync)
    {
        matrix(a), matrix(b);
        const int m = (int)a.size(0), k = (int)a.size(1), n = (int)b.size(0);
        const bool raw = !s_tok;
        require(a.scalar_type() == at::kChar && b.scalar_type() == at::kChar, "int8 operands");
        if (!raw)
            require(s_tok->scalar_type() == at::kFloat && s_ch->scalar_type() == at::kFloat, "fp32 scales");
        Output y(out, m, n, raw ? at::kInt : at::kHalf, a);
        const SyncPlan plan(sync);
        Workspace w(workspace, a, [&] {
            return plan.ptr ? nnf_w8a8_gemm_variant_workspace_bytes(m, n, k, NNF_W8A8_AUTO, plan.ptr) : nnf_w8a8_gemm_workspace_bytes(m, n, k);
        });
        call(plan.ptr ? "nnf_w8a8_gemm_variant" : raw ? "nnf_w8a8_gemm_acc" : "nnf_w8a8_gemm", nnf_w8a8_gemm_variant, stream(),
             a.data_ptr(), raw ? nullptr : s_tok->data_ptr(), b.data_ptr(), raw ? nullptr : s_ch->data_ptr(), raw ? nullptr : y.data,
             raw ? y.data : nullptr, m, n, k, NNF_W8A8_AUTO, plan.ptr, w.data, w.bytes);
        return y.release();
    }
    // (a, s_tok, w, s_ch, out, workspace, sync)
    PyObject* w8a8_gemm(Args v) { return w8a8(tensor(v[0]), tensor(v[2]), &tensor(v[1]), &tensor(v[3]), v[4], v[5], v[6]); }
    // (a, w, out, workspace, sync)
    PyObject* w8a8_gemm_acc(Args v) { return w8a8(tensor(v[0]), tensor(v[1]), nullptr, nullptr, v[2], v[3], v[4]); }

    // (op, a, b, out)
    PyObject* elementwise(Args v)
    {
        const Tensor& a = tensor(v[1]);
        require(a.scalar_type() == at::kHalf && a.is_contiguous(), "a contiguous fp16 tensor");
        const int64_t cols = a.size(-1);
        const size_t rows = cols ? (size_t)(a.numel() / cols) : 0;
        int b_is_row = 0;
        if (v[2] != Py_None)
        {
            const Tensor& b = tensor(v[2]);
            require(b.scalar_type() == at::kHalf && b.is_contiguous(), "a contiguous fp16 second operand");
            b_is_row = b.dim() == 1 && a.dim() > 1;
            require(b_is_row || b.sizes() == a.sizes(), "operands of one shape");
        }
        PyObject* out = v[3];
        if (out == Py_None)
        {
            out = THPVariable_Wrap(at::empty_like(a));
            if (!out)
                throw Raised();
        }
        else
            Py_INCREF(out);
        try
        {
            call("nnf_elementwise_f16", nnf_elementwise_f16, stream(), integer(v[0]), a.data_ptr(), address(v[2]), tensor(out).data_ptr(),
                 rows, (int)cols, b_is_row);
        }
        catch (...)
        {
            Py_DECREF(out);
            throw;
        }
        return out;
    }

    // (x, gamma, eps, out)
    PyObject* rms_norm(Args v)
    {
        const Tensor& x = tensor(v[0]);
        matrix(x);
        const int m = (int)x.size(0), k = (int)x.size(1);
        Output y(v[3], m, k, x.scalar_type(), x);
        call("nnf_rms_norm_f16", nnf_rms_norm_f16, stream(), x.data_ptr(), address(v[1]), y.data, m, k, real(v[2]));
        return y.release();
    }

    // (wq, scales, bits, group, zp, zero_points, out)
    PyObject* dequantize(Args v)
    {
        const Tensor& wq = tensor(v[0]);
        matrix(wq);
        const nnf_quant q = quant(v[2], v[3], v[4], v[5]);
        require(q.bits > 0, "bits of the weights");
        const int n = (int)wq.size(0), k = (int)(wq.size(1) * 8 / q.bits);
        Output y(v[6], n, k, at::kHalf, wq);
        call("nnf_dequantize_f16", nnf_dequantize_f16, stream(), wq.data_ptr(), address(v[1]), y.data, n, k, &q);
        return y.release();
    }

    template <PyObject* (*F)(Args), int N>
    PyObject* entry(PyObject*, Args v, Py_ssize_t n)
    {
        if (n != N)
        {
            PyErr_Format(PyExc_TypeError, "%d arguments expected, %zd given", N, n);
            return nullptr;
        }
        try
        {
            return F(v);
        }
        catch (const Raised&)
        {
        }
        catch (const std::exception& e)
        {
            PyErr_SetString(PyExc_RuntimeError, e.what());
        }
        return nullptr;
    }

    PyObject* set_error(PyObject*, PyObject* type)
    {
        Py_INCREF(type);
        Py_XDECREF(g_error);
        g_error = type;
        Py_RETURN_NONE;
    }

#define NNF_ENTRY(f, n) {#f, (PyCFunction)(void (*)(void))entry<f, n>, METH_FASTCALL, nullptr}
    PyMethodDef methods[] = {NNF_ENTRY(w4a16_gemm, 7),       NNF_ENTRY(wna16_gemm, 11),      NNF_ENTRY(w4a16_gemm_fused, 14), NNF_ENTRY(fused_mlp_w4a16, 13),
                             NNF_ENTRY(wna16_gemm_fused, 14), NNF_ENTRY(fused_mlp_wna16, 14), NNF_ENTRY(w8a8_gemm, 7),         NNF_ENTRY(w8a8_gemm_acc, 5),
                             NNF_ENTRY(elementwise, 4),       NNF_ENTRY(rms_norm, 4),         NNF_ENTRY(dequantize, 7),        {"set_error", set_error, METH_O, nullptr},
                             {nullptr, nullptr, 0, nullptr}};
    PyModuleDef module = {PyModuleDef_HEAD_INIT, "nnf_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
} // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit_nnf_torch()
{
    return PyModule_Create(&module);
}

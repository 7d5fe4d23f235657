// torch_binding.cpp -- the calls of minitensor_amd/__init__.py from torch
// tensors to the C ABI (include/mtgemm.h) without the interpreter in between:
// operand descriptors, outputs, workspace and launch in one native call.  The
// Python form of the same steps (three ctypes descriptors, two allocations, two
// foreign calls) took 13 us for a 256x512x512 product whose kernel takes 4.5.
//
// The interpreter lock is not held from the first allocation to the last launch,
// as it was not through the ctypes calls: a launch may wait for a full queue, and
// what it waits for (a host callback on the stream) may wait for the lock.
//
// Every function returns None where a call is not the plain case (an operand
// that is no fp32 tensor on a GPU, a wrapped or mismatched one): the caller then
// takes its own path, whose checks and errors are the contract.
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include "mtgemm.h"

namespace py = pybind11;

namespace {

// A plain fp32 tensor on a GPU with memory of its own.
bool plain(const at::Tensor& t) {
    return t.defined() && t.is_cuda() && t.scalar_type() == at::kFloat &&
           t.layout() == at::kStrided && t.has_storage() && !t.is_conj() && !t.is_neg() &&
           !t.unsafeGetTensorImpl()->is_python_dispatch();
}

// The tensor of a Python argument (nothing for None); `ok` is cleared for
// anything but a plain tensor.
at::Tensor arg(py::handle h, bool* ok) {
    if (h.is_none()) return {};
    if (!THPVariable_Check(h.ptr())) {
        *ok = false;
        return {};
    }
    at::Tensor t = THPVariable_Unpack(h.ptr());
    if (!plain(t)) *ok = false;
    return t;
}

const float* ptr(const at::Tensor& t) {
    return t.defined() ? static_cast<const float*>(t.data_ptr()) : nullptr;
}

mt_mat_f32 mat(const at::Tensor& t) {
    const bool b = t.dim() == 3;
    const int r = b ? 1 : 0;
    return mt_mat_f32{ptr(t), 0, t.size(r), t.size(r + 1), t.stride(r), t.stride(r + 1),
                      b ? t.size(0) : 1, b ? t.stride(0) : 0};
}

at::Tensor empty(at::IntArrayRef shape, const at::Tensor& like) {
    return at::empty(shape, at::TensorOptions().dtype(at::kFloat).device(like.device()));
}

// The caller's workspace, or one of `need` bytes.
struct Workspace {
    at::Tensor own;
    void* p = nullptr;
    size_t n = 0;
    template <class Need>
    Workspace(const at::Tensor& given, const at::Tensor& like, Need need) {
        if (given.defined()) {
            own = given;
            n = (size_t)own.numel();
        } else if ((n = need()) > 0) {
            own = at::empty({(int64_t)n}, at::TensorOptions().dtype(at::kByte).device(like.device()));
        }
        p = own.defined() ? own.data_ptr() : nullptr;
    }
};

// The caller's workspace (nothing for None); `ok` is cleared for no tensor.
at::Tensor given_ws(py::handle h, bool* ok) {
    if (h.is_none()) return {};
    if (THPVariable_Check(h.ptr())) return THPVariable_Unpack(h.ptr());
    *ok = false;
    return {};
}

void check(int rc, const char* what) {
    if (rc == MT_OK) return;
    const std::string msg =
        std::string(what) + ": " + mt_strerror(rc) + " (" + std::to_string(rc) + ")";
    if (rc == MT_ERR_INVALID) throw py::value_error(msg);
    throw std::runtime_error(msg);
}

// The stream given (its handle), or the current one of the current device.
void* stream_of(py::handle s) {
    return s.is_none() ? static_cast<void*>(c10::hip::getCurrentHIPStream().stream())
                       : reinterpret_cast<void*>(py::cast<uintptr_t>(s));
}

py::object tensor(const at::Tensor& t) {
    return t.defined() ? py::reinterpret_steal<py::object>(THPVariable_Wrap(t)) : py::none();
}

py::object gemm(py::handle pa, py::handle pb, py::handle pout, py::handle pbias, int axis,
                float beta, py::handle pws, py::handle stream) {
    bool ok = true;
    const at::Tensor gws = given_ws(pws, &ok);
    const at::Tensor a = arg(pa, &ok), b = arg(pb, &ok), bias = arg(pbias, &ok);
    at::Tensor out = arg(pout, &ok);
    if (!ok || !a.defined() || !b.defined()) return py::none();
    const int64_t d = a.dim();
    if ((d != 2 && d != 3) || b.dim() != d || a.size(d - 1) != b.size(d - 2) ||
        (bias.defined() && (axis == MT_BIAS_NONE || bias.dim() < 1)))
        return py::none();
    const int64_t m = a.size(d - 2), n = b.size(d - 1);
    const int64_t batch = d == 3 ? std::max(a.size(0), b.size(0)) : 1;
    if (out.defined() && (out.dim() != d || out.size(d - 2) != m || out.size(d - 1) != n ||
                          (d == 3 && out.size(0) != batch)))
        return py::none();
    void* const s = stream_of(stream);
    {
        const py::gil_scoped_release nogil;
        if (!out.defined()) out = d == 3 ? empty({batch, m, n}, a) : empty({m, n}, a);
        const mt_mat_f32 ma = mat(a), mb = mat(b), mc = mat(out);
        mt_epilogue_f32 ep{ptr(bias), bias.defined() ? bias.stride(-1) : 0,
                           bias.defined() ? axis : MT_BIAS_NONE, beta};
        const Workspace ws(gws, a, [&] { return mt_gemm_workspace_f32(&ma, &mb, &mc); });
        check(mt_gemm_f32(&ma, &mb, &mc, bias.defined() || beta != 0.f ? &ep : nullptr, ws.p, ws.n,
                          s),
              "mt_gemm_f32");
    }
    return pout.is_none() ? tensor(out) : py::reinterpret_borrow<py::object>(pout);
}

py::object linear(py::handle px, py::handle pw, py::handle pb, py::handle pout, py::handle pws,
                  py::handle stream) {
    bool ok = true;
    const at::Tensor gws = given_ws(pws, &ok);
    const at::Tensor x = arg(px, &ok), w = arg(pw, &ok), b = arg(pb, &ok);
    at::Tensor out = arg(pout, &ok);
    if (!ok || !x.defined() || !w.defined() || x.dim() != 2 || w.dim() != 2 ||
        x.size(1) != w.size(1) || (b.defined() && (b.dim() != 1 || b.size(0) != w.size(0))) ||
        (out.defined() && out.dim() != 2))
        return py::none();
    void* const s = stream_of(stream);
    {
        const py::gil_scoped_release nogil;
        if (!out.defined()) out = empty({x.size(0), w.size(0)}, x);
        const mt_mat_f32 mx = mat(x), mw = mat(w), my = mat(out);
        const Workspace ws(gws, x, [&] {
            return mt_linear_workspace_f32(x.size(0), x.size(1), w.size(0));
        });
        check(mt_linear_forward_f32(&mx, &mw, ptr(b), b.defined() ? b.stride(0) : 0, &my, ws.p,
                                    ws.n, s),
              "mt_linear_forward_f32");
    }
    return pout.is_none() ? tensor(out) : py::reinterpret_borrow<py::object>(pout);
}

py::object linear_backward(py::handle pdy, py::handle px, py::handle pw, bool need_dx,
                           bool need_dw, bool need_db, py::handle pdx, py::handle pdw,
                           py::handle pdb, float beta_w, float beta_b, py::handle pws,
                           py::handle stream) {
    bool ok = true;
    const at::Tensor gws = given_ws(pws, &ok);
    const at::Tensor dy = arg(pdy, &ok), x = arg(px, &ok), w = arg(pw, &ok);
    at::Tensor dx = arg(pdx, &ok), dw = arg(pdw, &ok), db = arg(pdb, &ok);
    if (!ok || !dy.defined() || !x.defined() || !w.defined() || dy.dim() != 2 || x.dim() != 2 ||
        w.dim() != 2 || (dx.defined() && dx.dim() != 2) || (dw.defined() && dw.dim() != 2) ||
        (db.defined() && db.dim() != 1))
        return py::none();
    const int64_t rows = x.size(0), fin = x.size(1), fout = w.size(0);
    void* const s = stream_of(stream);
    {
        const py::gil_scoped_release nogil;
        if (need_dx && !dx.defined()) dx = empty({rows, fin}, x);
        if (need_dw && !dw.defined()) dw = empty({fout, fin}, x);
        if (need_db && !db.defined()) db = empty({fout}, x);
        const mt_mat_f32 mdy = mat(dy), mx = mat(x), mw = mat(w);
        mt_mat_f32 mdx{}, mdw{};
        if (need_dx) mdx = mat(dx);
        if (need_dw) mdw = mat(dw);
        const Workspace ws(gws, x, [&] { return mt_linear_workspace_f32(rows, fin, fout); });
        check(mt_linear_backward_f32(&mdy, &mx, &mw, need_dx ? &mdx : nullptr,
                                     need_dw ? &mdw : nullptr, beta_w,
                                     need_db ? const_cast<float*>(ptr(db)) : nullptr,
                                     need_db ? db.stride(0) : 0, beta_b, ws.p, ws.n, s),
              "mt_linear_backward_f32");
    }
    const auto back = [](py::handle given, const at::Tensor& t) {
        return given.is_none() ? tensor(t) : py::reinterpret_borrow<py::object>(given);
    };
    return py::make_tuple(back(pdx, dx), back(pdw, dw), back(pdb, db));
}

py::object conv2d(py::handle px, py::handle pw, py::handle pb, int64_t stride, int64_t pad,
                  py::handle pws, py::handle stream) {
    bool ok = true;
    const at::Tensor gws = given_ws(pws, &ok);
    const at::Tensor x = arg(px, &ok);
    at::Tensor w = arg(pw, &ok), b = arg(pb, &ok);
    if (!ok || !x.defined() || !w.defined() || x.dim() != 4 || w.dim() != 4 ||
        x.size(1) != w.size(1) || !w.is_contiguous() || stride < 1 || pad < 0 ||
        w.size(2) < 1 || w.size(3) < 1 ||
        (b.defined() && (b.dim() != 1 || b.size(0) != w.size(0) || !b.is_contiguous())))
        return py::none();
    const mt_conv2d_desc d{x.size(0), x.size(1), x.size(2), x.size(3), w.size(0),
                           w.size(2), w.size(3), stride, pad};
    const auto extent = [&](int64_t in, int64_t k) {
        return in + 2 * pad < k ? 0 : (in + 2 * pad - k) / stride + 1;
    };
    void* const s = stream_of(stream);
    at::Tensor out;
    {
        const py::gil_scoped_release nogil;
        out = empty({d.n, d.c_out, extent(d.h, d.kh), extent(d.w, d.kw)}, x);
        const Workspace ws(gws, x, [&] { return mt_conv2d_workspace_f32(&d); });
        const int64_t st[4] = {x.stride(0), x.stride(1), x.stride(2), x.stride(3)};
        check(mt_conv2d_fwd_strided_f32(&d, ptr(x), st, ptr(w), ptr(b),
                                        const_cast<float*>(ptr(out)), ws.p, ws.n, s),
              "mt_conv2d_fwd_strided_f32");
    }
    return tensor(out);
}

py::object conv2d_backward(py::handle px, py::handle pw, py::handle pdy, int64_t stride,
                           int64_t pad, bool need_dx, bool need_dw, bool need_db,
                           py::handle pws, py::handle pdw, float beta_w, py::handle stream) {
    bool ok = true;
    const at::Tensor gws = given_ws(pws, &ok);
    const at::Tensor x = arg(px, &ok), w = arg(pw, &ok), dy = arg(pdy, &ok);
    at::Tensor dw = arg(pdw, &ok);
    if (!ok || !x.defined() || !w.defined() || !dy.defined() || x.dim() != 4 || w.dim() != 4 ||
        dy.dim() != 4 || !x.is_contiguous() || !w.is_contiguous() || !dy.is_contiguous() ||
        stride < 1 || pad < 0 || w.size(2) < 1 || w.size(3) < 1)
        return py::none();
    const mt_conv2d_desc d{x.size(0), x.size(1), x.size(2), x.size(3), w.size(0),
                           w.size(2), w.size(3), stride, pad};
    const auto extent = [&](int64_t in, int64_t k) {
        return in + 2 * pad < k ? 0 : (in + 2 * pad - k) / stride + 1;
    };
    if (dy.size(0) != d.n || dy.size(1) != d.c_out || dy.size(2) != extent(d.h, d.kh) ||
        dy.size(3) != extent(d.w, d.kw) ||
        (need_dw && dw.defined() && (dw.sizes() != w.sizes() || !dw.is_contiguous())))
        return py::none();
    void* const s = stream_of(stream);
    const auto out = [](const at::Tensor& t) { return const_cast<float*>(ptr(t)); };
    at::Tensor dx, db;
    {
        const py::gil_scoped_release nogil;
        const Workspace ws(gws, x, [&] { return mt_conv2d_bwd_workspace_f32(&d); });
        if (need_dx) {
            dx = empty(x.sizes(), x);
            check(mt_conv2d_bwd_input_f32(&d, ptr(dy), ptr(w), out(dx), ws.p, ws.n, s),
                  "mt_conv2d_bwd_input_f32");
        }
        if (need_db) db = empty({d.c_out}, x);
        if (need_dw) {
            if (!dw.defined()) dw = empty(w.sizes(), x);
            check(mt_conv2d_bwd_weight_bias_f32(&d, ptr(x), ptr(dy), out(dw), beta_w, out(db), 0.f,
                                                ws.p, ws.n, s),
                  "mt_conv2d_bwd_weight_bias_f32");
        } else if (need_db) {
            check(mt_conv2d_bwd_bias_f32(&d, ptr(dy), out(db), 0.f, s), "mt_conv2d_bwd_bias_f32");
        }
    }
    const py::object rdw = !need_dw          ? py::object(py::none())
                           : !pdw.is_none() ? py::reinterpret_borrow<py::object>(pdw)
                                            : tensor(dw);
    return py::make_tuple(tensor(dx), rdw, tensor(db));
}

}  // namespace

PYBIND11_MODULE(_native, m) {
    m.def("gemm", &gemm);
    m.def("linear", &linear);
    m.def("linear_backward", &linear_backward);
    m.def("conv2d", &conv2d);
    m.def("conv2d_backward", &conv2d_backward);
}

// Native bodies of the optimizer classes' step(): one call per parameter group
// walks the group's parameters, gradients and state and forwards to the C ABI.
// The lists that the `_ops.*_fused_step` functions take cost a Python loop over
// the parameters and one reference per tensor and list on the way in, 11 of the
// 18 us of host time of a Grokfast step on 14 tensors whose kernel takes 5 us.
//
// A call that meets anything but the ordinary case (state not created yet, a
// step counter that is no int) changes nothing and returns False; the class then
// takes its Python path, which creates the state and calls the list functions.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/profiler.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "ops_common.hpp"

namespace {

struct Member {
    const at::Tensor *p, *g;
    const at::Tensor* b[4];
    PyObject* state;
    long long step;
};

PyObject* name_of(const char* s) { return PyUnicode_InternFromString(s); }      // kept for the life of the process

const at::Tensor* as_tensor(PyObject* o) { return o && THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// Entry of optimizer.state for a parameter, or NULL.  torch's Tensor hashes by identity through a Python-level
// __hash__; the identity is tried first and the general lookup serves subclasses that hash otherwise.
PyObject* state_entry(PyObject* state, PyObject* param) {
    PyObject* e = _PyDict_GetItem_KnownHash(state, param, (Py_hash_t)(uintptr_t)param);
    if (!e) e = PyDict_GetItemWithError(state, param);
    if (!e) PyErr_Clear();
    return e;
}

// The group's parameters that have a non-empty gradient, with `n` state buffers each; steps counted up when `count`.
// False (and nothing changed) where the general path has to be taken.
bool gather(PyObject* params, PyObject* state, PyObject* const* names, int n, bool count, std::vector<Member>* out) {
    static PyObject* const kStep = name_of("step");
    if (!PyList_Check(params) || !PyDict_Check(state)) return false;
    const Py_ssize_t P = PyList_GET_SIZE(params);
    out->reserve(P);
    for (Py_ssize_t i = 0; i < P; i++) {
        PyObject* po = PyList_GET_ITEM(params, i);
        Member m;
        m.p = as_tensor(po);
        if (!m.p) return false;
        m.g = &m.p->grad();
        if (!m.g->defined()) continue;
        m.state = state_entry(state, po);
        if (!m.state || !PyDict_Check(m.state)) return false;
        for (int k = 0; k < n; k++) {
            m.b[k] = as_tensor(PyDict_GetItem(m.state, names[k]));
            if (!m.b[k]) return false;
        }
        m.step = 0;
        if (count) {
            PyObject* s = PyDict_GetItem(m.state, kStep);
            if (!s || !PyLong_CheckExact(s)) return false;
            m.step = PyLong_AsLongLong(s) + 1;
        }
        out->push_back(m);
    }
    if (count) {
        long long shared = -1;
        PyObject* value = nullptr;       // parameters of a group are nearly always at one step: one int object for all
        for (Member& m : *out) {
            if (m.step != shared) {
                Py_XDECREF(value);
                value = PyLong_FromLongLong(m.step);
                shared = m.step;
            }
            PyDict_SetItem(m.state, kStep, value);
        }
        Py_XDECREF(value);
    }
    return true;
}

void check_pair(const at::Tensor& p, const at::Tensor& g, const char* fn) {
    check_gpu(p, fn, "param");
    check_gpu(g, fn, "grad");
    TORCH_CHECK(p.scalar_type() == g.scalar_type(), fn, ": param/grad dtype mismatch");
    TORCH_CHECK(p.numel() == g.numel(), fn, ": param/grad size mismatch");
}
float* f32_ptr(const at::Tensor& t, int64_t n, const char* fn, const char* what) {
    check_f32(t, fn, what);
    TORCH_CHECK(t.numel() == n, fn, ": ", what, " size mismatch");
    return t.data_ptr<float>();
}

// per-step bias corrections, computed once for tensors at the same step
struct FloatCorrections {       // float pow, as the reference computes them (csrc/ops.cpp:333-334)
    float beta1, beta2, bc1 = 1.0f, bc2 = 1.0f;
    long long at = -1;
    void operator()(long long step) {
        if (step == at) return;
        at = step;
        bc1 = 1.0f - std::pow(beta1, static_cast<float>(step));
        bc2 = 1.0f - std::pow(beta2, static_cast<float>(step));
    }
};

struct Family {
    std::vector<SgFamilyTensor> ts;
    std::vector<int64_t> numels;
    const at::Tensor* first = nullptr;
    torch::Tensor ws;
    void add(const SgFamilyTensor& t, const at::Tensor* g) {
        ts.push_back(t);
        numels.push_back(t.numel);
        if (!first) first = g;
    }
    void make_ws() { ws = make_workspace(sg_family_workspace_bytes((int)ts.size(), numels.data()), *first); }
    void* stream() const { return current_stream(*first); }
};

// exp_avg, exp_avg_sq (n >= 2), aux (n >= 3), aux2 in fp32 (n >= 4), in the order the names were given
Family family_of(const std::vector<Member>& ms, int n, const char* fn) {
    Family F;
    F.ts.reserve(ms.size());
    F.numels.reserve(ms.size());
    for (const Member& m : ms) {
        if (m.g->numel() == 0) continue;
        check_pair(*m.p, *m.g, fn);
        SgFamilyTensor t = {};
        t.param = m.p->data_ptr();
        t.grad = m.g->data_ptr();
        t.numel = m.g->numel();
        t.dtype = dtype_code(*m.g, "grad");
        t.exp_avg = f32_ptr(*m.b[0], t.numel, fn, "exp_avg");
        if (n > 1) t.exp_avg_sq = f32_ptr(*m.b[1], t.numel, fn, "exp_avg_sq");
        if (n > 2) t.aux = f32_ptr(*m.b[2], t.numel, fn, "state");
        if (n > 3) t.aux2 = f32_ptr(*m.b[3], t.numel, fn, "param_init");
        t.bc1 = t.bc2 = 1.0f;
        F.add(t, m.g);
    }
    return F;
}
// (members with an empty gradient are skipped by family_of: the corrections follow the same rule)
template <class C>
void correct(Family* F, const std::vector<Member>& ms, C corr) {
    size_t k = 0;
    for (const Member& m : ms) {
        if (m.g->numel() == 0) continue;
        corr(m.step);
        F->ts[k].bc1 = corr.bc1;
        F->ts[k].bc2 = corr.bc2;
        k++;
    }
}

bool grokfast_group_step(py::handle params, py::handle state, float alpha, float lamb, double lr, double beta1, double beta2, double eps,
                         double weight_decay) {
    const char* fn = "grokfast_adamw_fused_step";
    static PyObject* const names[3] = {name_of("ema"), name_of("exp_avg"), name_of("exp_avg_sq")};
    std::vector<Member> ms;
    if (!gather(params.ptr(), state.ptr(), names, 3, true, &ms)) return false;
    std::vector<SgGrokfastAdamTensor> ts;
    std::vector<int64_t> numels;
    ts.reserve(ms.size());
    numels.reserve(ms.size());
    const at::Tensor* first = nullptr;
    for (const Member& m : ms) {
        const int64_t n = m.g->numel();
        if (n == 0) continue;
        check_pair(*m.p, *m.g, fn);
        ts.push_back({m.p->data_ptr(), m.g->data_ptr(), f32_ptr(*m.b[0], n, fn, "ema_buf"), f32_ptr(*m.b[1], n, fn, "exp_avg"),
                      f32_ptr(*m.b[2], n, fn, "exp_avg_sq"), n, dtype_code(*m.g, "grad"), (int32_t)m.step});
        numels.push_back(n);
        if (!first) first = m.g;
    }
    if (ts.empty()) return true;
    torch::Tensor ws;
    if (ts.size() > SG_ELEMWISE_ARG_TENSORS) ws = make_workspace(sg_elemwise_workspace_bytes((int)ts.size(), numels.data()), *first);
    check_status(sg_grokfast_adamw_step((int)ts.size(), ts.data(), alpha, lamb, lr, beta1, beta2, eps, weight_decay,
                                        ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? (size_t)ws.numel() : 0, current_stream(*first)),
                 fn);
    return true;
}

bool lion_group_step(py::handle params, py::handle state, float lr, float beta1, float beta2, float wd) {
    static PyObject* const names[1] = {name_of("exp_avg")};
    std::vector<Member> ms;
    if (!gather(params.ptr(), state.ptr(), names, 1, false, &ms)) return false;
    Family F = family_of(ms, 1, "lion_fused_step");
    if (F.ts.empty()) return true;
    const bool ws = F.ts.size() > SG_ELEMWISE_ARG_TENSORS;
    if (ws) F.make_ws();
    check_status(sg_lion_step((int)F.ts.size(), F.ts.data(), lr, beta1, beta2, wd, ws ? F.ws.data_ptr() : nullptr,
                              ws ? (size_t)F.ws.numel() : 0, F.stream()), "lion_fused_step");
    return true;
}

bool grokadamw_group_step(py::handle params, py::handle state, float alpha, float lamb, float beta1, float beta2, float lr, float wd,
                          float eps, float grad_clip_norm) {
    static PyObject* const names[3] = {name_of("exp_avg"), name_of("exp_avg_sq"), name_of("ema")};
    std::vector<Member> ms;
    if (!gather(params.ptr(), state.ptr(), names, 3, true, &ms)) return false;
    Family F = family_of(ms, 3, "grokadamw_fused_step");
    if (F.ts.empty()) return true;
    correct(&F, ms, FloatCorrections{beta1, beta2});
    F.make_ws();
    check_status(sg_grokadamw_step((int)F.ts.size(), F.ts.data(), alpha, lamb, beta1, beta2, lr, wd, eps, grad_clip_norm, F.ws.data_ptr(),
                                   (size_t)F.ws.numel(), F.stream()), "grokadamw_fused_step");
    return true;
}

// AdamW with bias corrections in double (adamw_step of _adamw_helper.py)
struct DoubleCorrections {
    double beta1, beta2;
    float bc1 = 1.0f, bc2 = 1.0f;
    long long at = -1;
    void operator()(long long step) {
        if (step == at) return;
        at = step;
        bc1 = (float)(1.0 - std::pow(beta1, (double)step));
        bc2 = (float)(1.0 - std::pow(beta2, (double)step));
    }
};
bool adamw_group_step(py::handle params, py::handle state, double lr, double beta1, double beta2, double eps, double wd) {
    static PyObject* const names[2] = {name_of("exp_avg"), name_of("exp_avg_sq")};
    std::vector<Member> ms;
    if (!gather(params.ptr(), state.ptr(), names, 2, true, &ms)) return false;
    Family F = family_of(ms, 2, "adamw_fused_step");
    if (F.ts.empty()) return true;
    correct(&F, ms, DoubleCorrections{beta1, beta2});
    const bool ws = F.ts.size() > SG_ELEMWISE_ARG_TENSORS;
    if (ws) F.make_ws();
    check_status(sg_grokadamw_step((int)F.ts.size(), F.ts.data(), 0.0f, 0.0f, (float)beta1, (float)beta2, (float)lr, (float)wd, (float)eps,
                                   0.0f, ws ? F.ws.data_ptr() : nullptr, ws ? (size_t)F.ws.numel() : 0, F.stream()), "adamw_fused_step");
    return true;
}

// The amplifier's four tensors on `device`, for an amplifier that lives on the CPU: one packed copy per device, made again
// whenever the values differ from those it was made from (a comparison of a few hundred floats takes 0.1 us, a copy 20 us;
// version counters do not see writes through .data or a NumPy view).  The copy is complete before it is handed out, and a
// stream other than the one it was made on is recorded with it, so that replacing it does not free it under that
// stream's kernels; a graph that captures its address keeps it for good.
py::tuple amplifier_on(const std::vector<torch::Tensor>& weights, py::dict held, const torch::Device& device) {
    int64_t total = 0;
    for (const torch::Tensor& w : weights) {
        TORCH_CHECK(w.device().is_cpu() && w.scalar_type() == torch::kFloat32 && w.is_contiguous(), "amplifier weights must be contiguous float32 on the CPU");
        total += w.numel();
    }
    const auto stream = c10::hip::getCurrentHIPStream(device.index());
    const py::int_ key(stream.device_index()), made_on((uintptr_t)stream.stream());
    if (held.contains(key)) {
        const py::tuple entry = held[key];
        const torch::Tensor made_from = entry[0].cast<torch::Tensor>();
        bool same = made_from.numel() == total;
        int64_t o = 0;
        for (const torch::Tensor& w : weights) {
            same = same && std::memcmp(made_from.data_ptr<float>() + o, w.data_ptr<float>(), sizeof(float) * (size_t)w.numel()) == 0;
            o += w.numel();
        }
        if (same) {
            if (!py::object(entry[3]).equal(made_on))
                entry[1].cast<torch::Tensor>().record_stream(c10::Stream(c10::Stream::UNSAFE, device, stream.id()));
            hipStreamCaptureStatus status = hipStreamCaptureStatusNone;      // (the null stream cannot capture)
            if (stream.stream() != nullptr && hipStreamIsCapturing(stream.stream(), &status) == hipSuccess && status != hipStreamCaptureStatusNone) {
                if (!held.contains("captured")) held["captured"] = py::list();
                held["captured"].cast<py::list>().append(entry[1]);
            }
            return entry[2].cast<py::tuple>();
        }
    }
    at::NoGradGuard guard;
    torch::Tensor host = torch::empty({total}, torch::kFloat32);
    int64_t o = 0;
    for (const torch::Tensor& w : weights) {
        std::memcpy(host.data_ptr<float>() + o, w.data_ptr<float>(), sizeof(float) * (size_t)w.numel());
        o += w.numel();
    }
    const torch::Tensor flat = host.to(device);
    py::tuple parts(weights.size());
    o = 0;
    for (size_t k = 0; k < weights.size(); k++) {
        parts[k] = py::cast(flat.narrow(0, o, weights[k].numel()).view(weights[k].sizes()));
        o += weights[k].numel();
    }
    held[key] = py::make_tuple(host, flat, parts, made_on);
    return parts;
}

bool neuralgrok_group_step(py::handle params, py::handle state, const torch::Tensor& W1, const torch::Tensor& b1, const torch::Tensor& W2,
                           const torch::Tensor& b2, float alpha_amp, float beta_amp, int hidden_dim, float beta1, float beta2, float lr,
                           float wd, float eps, float grad_clip_norm) {
    const char* fn = "neuralgrok_fused_step";
    static PyObject* const names[2] = {name_of("exp_avg"), name_of("exp_avg_sq")};
    std::vector<Member> ms;
    if (!gather(params.ptr(), state.ptr(), names, 2, true, &ms)) return false;
    Family F = family_of(ms, 2, fn);
    if (F.ts.empty()) return true;
    correct(&F, ms, FloatCorrections{beta1, beta2});
    check_f32(W1, fn, "W1"); check_f32(b1, fn, "b1"); check_f32(W2, fn, "W2"); check_f32(b2, fn, "b2");
    TORCH_CHECK(W1.numel() == hidden_dim && b1.numel() == hidden_dim && W2.numel() == hidden_dim && b2.numel() == 1, fn,
                ": amplifier weight shapes do not match hidden_dim");
    SgAmplifier amp = {W1.data_ptr<float>(), b1.data_ptr<float>(), W2.data_ptr<float>(), b2.data_ptr<float>(), hidden_dim};
    F.make_ws();
    check_status(sg_neuralgrok_step((int)F.ts.size(), F.ts.data(), &amp, alpha_amp, beta_amp, beta1, beta2, lr, wd, eps, grad_clip_norm,
                                    F.ws.data_ptr(), (size_t)F.ws.numel(), F.stream()), fn);
    return true;
}

// the new d_lr, or None where the general path has to be taken
py::object prodigy_group_step(py::handle params, py::handle state, float d_lr, float beta1, float beta2, float lr, float wd, float eps) {
    static PyObject* const names[4] = {name_of("exp_avg"), name_of("exp_avg_sq"), name_of("s"), name_of("param_init")};
    std::vector<Member> ms;
    if (!gather(params.ptr(), state.ptr(), names, 4, true, &ms)) return py::none();
    Family F = family_of(ms, 4, "prodigy_fused_step");
    if (F.ts.empty()) return py::float_(d_lr);
    correct(&F, ms, FloatCorrections{beta1, beta2});
    F.make_ws();
    float out = d_lr;
    check_status(sg_prodigy_step((int)F.ts.size(), F.ts.data(), d_lr, beta1, beta2, lr, wd, eps, &out, F.ws.data_ptr(), (size_t)F.ws.numel(),
                                 F.stream()), "prodigy_fused_step");
    return py::float_(out);
}

bool muon_group_step(py::handle params, py::handle state, float momentum, float lr, float wd, int ns_steps) {
    const char* fn = "muon_fused_step";
    static PyObject* const names[1] = {name_of("momentum_buffer")};
    std::vector<Member> ms;
    if (!gather(params.ptr(), state.ptr(), names, 1, false, &ms)) return false;
    std::vector<SgMuonMatrix> mats;
    mats.reserve(ms.size());
    const at::Tensor* first = nullptr;
    for (const Member& m : ms) {
        if (m.g->numel() == 0) continue;
        check_pair(*m.p, *m.g, fn);
        TORCH_CHECK(m.p->dim() == 2, fn, ": parameters must be 2-D");
        mats.push_back({m.p->data_ptr(), m.g->data_ptr(), f32_ptr(*m.b[0], m.p->numel(), fn, "momentum buffer"), m.p->size(0), m.p->size(1),
                        dtype_code(*m.p, "param")});
        if (!first) first = m.p;
    }
    if (mats.empty()) return true;
    auto ws = make_workspace(sg_muon_workspace_bytes((int)mats.size(), mats.data()), *first);
    check_status(sg_muon_step((int)mats.size(), mats.data(), momentum, lr, wd, ns_steps, ws.data_ptr(), (size_t)ws.numel(),
                              current_stream(*first)), fn);
    return true;
}

// ---- SuperGrok v1.5 / v1.1: flat lists, one entry per parameter of the optimizer ---------------
struct FlatLists {
    PyObject *params, *data, *ea, *easq, *mu, *sharp, *steps, *factors, *beta1s;
    Py_ssize_t n;
    bool ok() const {
        for (PyObject* l : {params, data, ea, easq, mu, sharp, steps, factors, beta1s})
            if (!PyList_Check(l) || PyList_GET_SIZE(l) != n) return false;
        return true;
    }
    const at::Tensor& at(PyObject* list, Py_ssize_t i) const {
        const at::Tensor* t = as_tensor(PyList_GET_ITEM(list, i));
        TORCH_CHECK(t, "optimizer state list holds a non-tensor");
        return *t;
    }
};
// sharpness is kept in fp32: the kernel rounds it to the gradient's type as it reads it
int sharp_code(const at::Tensor& sharp, const at::Tensor& g, const char* fn) {
    check_gpu(sharp, fn, "sharpness");
    TORCH_CHECK(sharp.numel() == g.numel(), fn, ": sharpness size mismatch");
    const int code = dtype_code(g, "grad");
    if (sharp.scalar_type() == g.scalar_type()) return code;
    TORCH_CHECK(sharp.scalar_type() == torch::kFloat32, fn, ": sharpness must be float32 or have the gradient's dtype");
    return code | SG_SHARP_F32;
}
struct NetArgs {
    torch::Tensor t[4];
    Sg15Net net;
    NetArgs(const torch::Tensor& W1, const torch::Tensor& b1, const torch::Tensor& W2, const torch::Tensor& b2, int hidden, float rescale,
            const char* fn) {
        const torch::Tensor* in[4] = {&W1, &b1, &W2, &b2};
        for (int k = 0; k < 4; k++) {
            t[k] = in[k]->to(torch::kFloat32).contiguous();
            check_f32(t[k], fn, "meta-net weight");
        }
        TORCH_CHECK(W1.numel() == 2 * hidden && b1.numel() == hidden && W2.numel() == hidden && b2.numel() == 1, fn,
                    ": meta-net weight shapes do not match hidden_dim");
        net = {t[0].data_ptr<float>(), t[1].data_ptr<float>(), t[2].data_ptr<float>(), t[3].data_ptr<float>(), hidden, rescale,
               g_sg15_gelu_mode};
    }
};
// calls f(i, grad, alpha_i, beta1_i, bc1, bc2) for every parameter with a non-empty gradient
template <class F>
void each_flat(const FlatLists& L, double alpha, float beta2, F f) {
    for (Py_ssize_t i = 0; i < L.n; i++) {
        const at::Tensor& g = L.at(L.params, i).grad();
        if (!g.defined() || g.numel() == 0) continue;
        // the step counters go into the call by value, as in the reference: a call counts its own copy up
        const float step = static_cast<float>(PyLong_AsLongLong(PyList_GET_ITEM(L.steps, i)) + 1);
        const double a = std::max(0.0, std::min(1.0, alpha * PyFloat_AsDouble(PyList_GET_ITEM(L.factors, i))));
        const float b1 = (float)PyFloat_AsDouble(PyList_GET_ITEM(L.beta1s, i));
        if (PyErr_Occurred()) throw py::error_already_set();
        f(i, g, (float)a, b1, 1.0f - std::pow(b1, step), 1.0f - std::pow(beta2, step));
    }
}

bool supergrok15_flat_step(py::handle params, py::handle data, py::handle eas, py::handle easqs, py::handle mus, py::handle sharps,
                           py::handle steps, double alpha, py::handle alpha_factors, py::handle beta1s, const torch::Tensor& W1,
                           const torch::Tensor& b1, const torch::Tensor& W2, const torch::Tensor& b2, float rescale, int hidden, float beta2,
                           float lr, float wd_eff, float eps, float lamb, float ramp, float gate_signal, float grad_clip_norm) {
    const char* fn = "supergrok15_fused_step";
    const FlatLists L = {params.ptr(), data.ptr(), eas.ptr(), easqs.ptr(), mus.ptr(), sharps.ptr(), steps.ptr(), alpha_factors.ptr(),
                         beta1s.ptr(), PyList_Check(params.ptr()) ? PyList_GET_SIZE(params.ptr()) : -1};
    if (!L.ok()) return false;
    std::vector<Sg15Tensor> ts;
    std::vector<int64_t> numels;
    ts.reserve(L.n);
    numels.reserve(L.n);
    const at::Tensor* first = nullptr;
    each_flat(L, alpha, beta2, [&](Py_ssize_t i, const at::Tensor& g, float a, float be, float bc1, float bc2) {
        const at::Tensor& p = L.at(L.data, i);
        check_pair(p, g, fn);
        const int64_t n = g.numel();
        const at::Tensor& s = L.at(L.sharp, i);
        ts.push_back({p.data_ptr(), g.data_ptr(), s.data_ptr(), f32_ptr(L.at(L.ea, i), n, fn, "exp_avg"),
                      f32_ptr(L.at(L.easq, i), n, fn, "exp_avg_sq"), f32_ptr(L.at(L.mu, i), n, fn, "mu"), n, sharp_code(s, g, fn), a, be,
                      bc1, bc2});
        numels.push_back(n);
        if (!first) first = &p;
    });
    if (ts.empty()) return true;
    const NetArgs N(W1, b1, W2, b2, hidden, rescale, fn);
    const float lamb_eff = ramp > 0.0f ? ramp * gate_signal * lamb : 0.0f;
    auto ws = make_workspace(sg_elemwise_workspace_bytes((int)ts.size(), numels.data()), *first);
    check_status(sg15_fused_step((int)ts.size(), ts.data(), &N.net, lamb_eff, beta2, lr, wd_eff, eps, grad_clip_norm, ws.data_ptr(),
                                 (size_t)ws.numel(), current_stream(*first)), fn);
    return true;
}

bool supergrok11_flat_step(py::handle params, py::handle data, py::handle eas, py::handle easqs, py::handle mus, py::handle sharps,
                           py::handle steps, double alpha, py::handle alpha_factors, py::handle beta1s, const torch::Tensor& W1,
                           const torch::Tensor& b1, const torch::Tensor& W2, const torch::Tensor& b2, float rescale, int hidden, float beta2,
                           float lr, float wd_eff, float eps, float lamb, float ramp, float gate_temperature, float grad_clip_norm) {
    const char* fn = "supergrok11_fused_step";
    const FlatLists L = {params.ptr(), data.ptr(), eas.ptr(), easqs.ptr(), mus.ptr(), sharps.ptr(), steps.ptr(), alpha_factors.ptr(),
                         beta1s.ptr(), PyList_Check(params.ptr()) ? PyList_GET_SIZE(params.ptr()) : -1};
    if (!L.ok()) return false;
    Family F;
    each_flat(L, alpha, beta2, [&](Py_ssize_t i, const at::Tensor& g, float a, float be, float bc1, float bc2) {
        const at::Tensor& p = L.at(L.data, i);
        check_pair(p, g, fn);
        const at::Tensor& s = L.at(L.sharp, i);
        SgFamilyTensor t = {};
        t.numel = g.numel();
        t.dtype = sharp_code(s, g, fn);
        t.param = p.data_ptr();
        t.grad = g.data_ptr();
        t.aux2 = s.data_ptr();
        t.exp_avg = f32_ptr(L.at(L.ea, i), t.numel, fn, "exp_avg");
        t.exp_avg_sq = f32_ptr(L.at(L.easq, i), t.numel, fn, "exp_avg_sq");
        t.aux = f32_ptr(L.at(L.mu, i), t.numel, fn, "mu");
        t.bc1 = bc1; t.bc2 = bc2; t.alpha = a; t.beta1 = be;
        F.add(t, &p);
    });
    if (F.ts.empty()) return true;
    const NetArgs N(W1, b1, W2, b2, hidden, rescale, fn);
    F.make_ws();
    check_status(sg11_fused_step((int)F.ts.size(), F.ts.data(), &N.net, beta2, lr, wd_eff, eps, lamb, ramp, gate_temperature, grad_clip_norm,
                                 F.ws.data_ptr(), (size_t)F.ws.numel(), F.stream()), fn);
    return true;
}

// ---- SuperGrok v2 ------------------------------------------------------------------------------
// The clip pre-pass and the batched step for every parameter with a gradient, step counters counted up in place.
// dims: d_model, d_state, d_inner, gru_hidden, num_heads, pk_dim, expert_hidden, num_experts.  Returns how many
// parameters took part, or -1 (nothing changed) where the general path has to be taken: a Mamba state that is not there
// yet, a gradient that is not contiguous, parameters elsewhere than on the GPU.
int64_t supergrok2_flat_step(py::list params, py::list eas, py::list easqs, py::list mus, py::list sharps, py::list grus, py::list mfwd,
                             py::list mbwd, py::list steps, double alpha, py::list alpha_factors, py::list beta1s, double lamb_eff,
                             py::list weights, float rescale, double beta2, float lr, float wd_eff, float eps, std::vector<int> dims8,
                             const torch::Tensor& expert_counts, double max_norm) {
    const char* fn = "supergrok2_mamba_peer_batched_step";
    const Py_ssize_t P = PyList_GET_SIZE(params.ptr());
    for (PyObject* l : {eas.ptr(), easqs.ptr(), mus.ptr(), sharps.ptr(), grus.ptr(), mfwd.ptr(), mbwd.ptr(), steps.ptr(), alpha_factors.ptr(),
                        beta1s.ptr()})
        if (PyList_GET_SIZE(l) != P) return -1;
    if (!(max_norm > 0.0) || dims8.size() != 8 || PyList_GET_SIZE(weights.ptr()) != SG2_NUM_WEIGHTS) return -1;
    const SgDims dims = {dims8[0], dims8[1], dims8[2], dims8[3], dims8[4], dims8[5], dims8[6], dims8[7]};
    auto item = [](const py::list& l, Py_ssize_t i) { return as_tensor(PyList_GET_ITEM(l.ptr(), i)); };
    std::vector<Sg2Tensor> ts;
    std::vector<int64_t> numels;
    std::vector<Py_ssize_t> active;
    ts.reserve(P);
    numels.reserve(P);
    active.reserve(P);
    const at::Tensor* first = nullptr;
    double bc2 = 1.0;
    long long bc2_at = -1;
    for (Py_ssize_t i = 0; i < P; i++) {
        const at::Tensor* p = item(params, i);
        if (!p) return -1;
        const at::Tensor& g = p->grad();
        if (!g.defined()) continue;
        const at::Tensor *ea = item(eas, i), *easq = item(easqs, i), *mu = item(mus, i), *s = item(sharps, i), *gru = item(grus, i),
                         *mf = item(mfwd, i), *mb = item(mbwd, i);
        PyObject* step = PyList_GET_ITEM(steps.ptr(), i);
        if (!ea || !easq || !mu || !s || !gru || !mf || !mb || !PyLong_CheckExact(step) || !p->is_cuda() || !g.is_cuda() ||
            !g.is_contiguous())
            return -1;
        active.push_back(i);
        const int64_t n = g.numel();
        if (n == 0) continue;
        const long long t = PyLong_AsLongLong(step) + 1;
        const double b1 = PyFloat_AsDouble(PyList_GET_ITEM(beta1s.ptr(), i));
        const double a = std::max(0.0, std::min(1.0, alpha * PyFloat_AsDouble(PyList_GET_ITEM(alpha_factors.ptr(), i))));
        if (PyErr_Occurred()) throw py::error_already_set();
        if (t != bc2_at) {
            bc2 = 1.0 - std::pow(beta2, (double)t);
            bc2_at = t;
        }
        check_pair(*p, g, fn);
        Sg2Tensor q = {};
        q.param = p->data_ptr();
        q.grad = g.data_ptr();
        q.sharpness = s->data_ptr();
        q.dtype = sharp_code(*s, g, fn);
        q.numel = n;
        q.exp_avg = f32_ptr(*ea, n, fn, "exp_avg");
        q.exp_avg_sq = f32_ptr(*easq, n, fn, "exp_avg_sq");
        q.mu = f32_ptr(*mu, n, fn, "mu");
        q.gru_state = f32_ptr(*gru, n * dims.gru_hidden, fn, "gru_state");
        q.mamba_fwd_state = f32_ptr(*mf, (int64_t)dims.d_inner * dims.d_state, fn, "mamba_fwd_state");
        q.mamba_bwd_state = f32_ptr(*mb, (int64_t)dims.d_inner * dims.d_state, fn, "mamba_bwd_state");
        q.alpha_mu = (float)a;
        q.lamb_eff = (float)lamb_eff;
        q.beta1 = (float)b1;
        q.bc1 = (float)(1.0 - std::pow(b1, (double)t));
        q.bc2 = (float)bc2;
        ts.push_back(q);
        numels.push_back(n);
        if (!first) first = p;
    }
    if (active.empty()) return 0;
    if (!first) return -1;
    const torch::Tensor* w[SG2_NUM_WEIGHTS];
    for (int k = 0; k < SG2_NUM_WEIGHTS; k++) {
        w[k] = item(weights, k);
        TORCH_CHECK(w[k], fn, ": meta-net weight ", k, " is no tensor");
    }
    Sg2Weights W;
    check_sg2_weights(fn, w, dims, &W);
    check_gpu(expert_counts, fn, "expert_counts");
    TORCH_CHECK(expert_counts.scalar_type() == torch::kInt32 && expert_counts.numel() == dims.num_experts, fn,
                ": expert_counts must be int32[num_experts]");
    const size_t bytes = sg2_workspace_bytes(&dims, (int)ts.size(), numels.data());
    TORCH_CHECK(bytes > 0, fn, ": ", sg_last_error());
    auto ws = make_workspace(bytes, *first);
    const Sg2Scalars sc = {rescale, (float)beta2, lr, wd_eff, eps};
    check_status(sg2_clipped_step(&dims, &W, (int)ts.size(), ts.data(), &sc, (float)max_norm, expert_counts.data_ptr<int32_t>(), ws.data_ptr(),
                                  (size_t)ws.numel(), current_stream(*first)), fn);
    for (Py_ssize_t i : active) {
        PyObject* next = PyLong_FromLongLong(PyLong_AsLongLong(PyList_GET_ITEM(steps.ptr(), i)) + 1);
        PyList_SetItem(steps.ptr(), i, next);
    }
    return (int64_t)active.size();
}

// The bilevel pass over tensors that stay where they are.  begin (sort and scan) returns what finish needs, or None where the
// general path has to be taken (other sizes of the net, tensors that would have to be converted).
struct BilevelPass {
    SgDims dims;
    Sg2Weights W;
    std::vector<Sg2Tensor> ts;
    std::vector<Py_ssize_t> at;            // the lists' index of each
    std::vector<at::Tensor> kept;          // whatever the records point to
    torch::Tensor ws;
    int64_t total = 0;
};

// exact: fp32 sharpness next to 16-bit gradients is used as it is
py::object supergrok2_bilevel_begin(py::list grads, py::list sharps, py::list grus, py::list mfwd, py::list mbwd, py::list weights, bool exact,
                                    std::vector<int> dims8) {
    const char* fn = "supergrok2_bilevel_begin";
    const Py_ssize_t P = PyList_GET_SIZE(grads.ptr());
    for (PyObject* l : {sharps.ptr(), grus.ptr(), mfwd.ptr(), mbwd.ptr()})
        if (PyList_GET_SIZE(l) != P) return py::none();
    if (P == 0 || dims8.size() != 8 || PyList_GET_SIZE(weights.ptr()) != SG2_NUM_WEIGHTS) return py::none();
    auto pass = std::make_unique<BilevelPass>();
    const SgDims dims = {dims8[0], dims8[1], dims8[2], dims8[3], dims8[4], dims8[5], dims8[6], dims8[7]};
    pass->dims = dims;
    auto item = [](const py::list& l, Py_ssize_t i) { return as_tensor(PyList_GET_ITEM(l.ptr(), i)); };
    std::vector<int64_t> numels;
    pass->kept.reserve(5 * P + SG2_NUM_WEIGHTS);
    for (Py_ssize_t i = 0; i < P; i++) {
        const at::Tensor *g = item(grads, i), *s = item(sharps, i), *gru = item(grus, i), *mf = item(mfwd, i), *mb = item(mbwd, i);
        if (!g || !s || !gru || !mf || !mb) return py::none();
        const int64_t n = g->numel();
        if (n == 0) continue;
        if (s->numel() != n || gru->numel() != n * dims.gru_hidden || mf->numel() != (int64_t)dims.d_inner * dims.d_state ||
            mb->numel() != mf->numel())
            return py::none();
        for (const at::Tensor* t : {g, s, gru, mf, mb}) {
            if (!t->is_cuda() || !t->is_contiguous()) return py::none();
            pass->kept.push_back(*t);
        }
        for (const at::Tensor* t : {gru, mf, mb})
            if (t->scalar_type() != torch::kFloat32) return py::none();
        if (((uintptr_t)gru->data_ptr() & 15u) != 0) return py::none();
        Sg2Tensor q = {};
        q.dtype = dtype_code(*g, "grad");
        if (s->scalar_type() != g->scalar_type()) {
            if (!exact || s->scalar_type() != torch::kFloat32) return py::none();
            q.dtype |= SG_SHARP_F32 | SG_SHARP_EXACT;
        }
        q.grad = g->data_ptr();
        q.sharpness = s->data_ptr();
        q.gru_state = gru->data_ptr<float>();
        q.mamba_fwd_state = mf->data_ptr<float>();
        q.mamba_bwd_state = mb->data_ptr<float>();
        q.numel = n;
        pass->ts.push_back(q);
        pass->at.push_back(i);
        numels.push_back(n);
        pass->total += n;
    }
    if (pass->ts.empty()) return py::none();
    const at::Tensor like = pass->kept[0];
    const torch::Tensor* w[SG2_NUM_WEIGHTS];
    for (int k = 0; k < SG2_NUM_WEIGHTS; k++) {
        w[k] = item(weights, k);
        if (!w[k]) return py::none();
        pass->kept.push_back(*w[k]);
    }
    check_sg2_weights(fn, w, dims, &pass->W);
    const size_t bytes = sg2_bilevel_pass_workspace_bytes(&dims, (int)pass->ts.size(), numels.data());
    TORCH_CHECK(bytes > 0, fn, ": ", sg_last_error());
    pass->ws = make_workspace(bytes, like);
    check_status(sg2_bilevel_pass_begin(&dims, &pass->W, (int)pass->ts.size(), pass->ts.data(), pass->ws.data_ptr(), (size_t)pass->ws.numel(),
                                        current_stream(like)), fn);
    return py::cast(std::move(pass));
}

// (smart gradients or None, gradients of the per-element weights, gradients of the scan weights), flat; normalise: the
// cotangent is -v / |v|.  None where a cotangent is not of its gradient's size and type.
py::object supergrok2_bilevel_finish(BilevelPass& pass, py::list cots, float rescale, bool normalise, bool want_smart) {
    const char* fn = "supergrok2_bilevel_finish";
    at::NoGradGuard guard;
    const Py_ssize_t given = PyList_GET_SIZE(cots.ptr());
    std::vector<at::Tensor> v;
    for (size_t k = 0; k < pass.ts.size(); k++) {
        const at::Tensor* c = pass.at[k] < given ? as_tensor(PyList_GET_ITEM(cots.ptr(), pass.at[k])) : nullptr;
        if (!c || !c->is_cuda() || c->numel() != pass.ts[k].numel || dtype_code(*c, "cotangent") != (pass.ts[k].dtype & ~(SG_SHARP_F32 | SG_SHARP_EXACT)))
            return py::none();
        v.push_back(c->contiguous());
        pass.ts[k].param = v.back().data_ptr();
    }
    const auto opt = torch::TensorOptions().device(pass.ws.device()).dtype(torch::kFloat32);
    torch::Tensor norms;
    // (tensor by tensor with the framework's own reduction, as v.norm() forms them: the sums of a fresh meta-net's experts can
    // nearly cancel, and the first step of an optimizer that divides by their size shows the last bits of the cotangents)
    if (normalise) {
        norms = torch::empty({(int64_t)v.size()}, opt);
        for (size_t i = 0; i < v.size(); i++) {
            at::Tensor out = norms.select(0, i);
            at::linalg_vector_norm_out(out, v[i].scalar_type() == torch::kFloat32 ? v[i] : v[i].to(torch::kFloat32), 2);
        }
    }
    auto elem = torch::empty({(SG2_ELEM_GRAD_FLOATS - pass.dims.num_experts * 49) + pass.dims.num_experts * (3 * pass.dims.expert_hidden + 1)}, opt);
    auto scan = torch::empty({SG2_SCAN_GRAD_FLOATS}, opt);
    torch::Tensor smart;
    if (want_smart) smart = torch::empty({pass.total}, opt);
    check_status(sg2_bilevel_pass_finish(&pass.dims, &pass.W, (int)pass.ts.size(), pass.ts.data(), rescale, normalise ? norms.data_ptr<float>() : nullptr,
                                         want_smart ? smart.data_ptr<float>() : nullptr, elem.data_ptr<float>(), scan.data_ptr<float>(),
                                         pass.ws.data_ptr(), (size_t)pass.ws.numel(), current_stream(pass.ws)), fn);
    return py::make_tuple(want_smart ? py::cast(smart) : py::object(py::none()), elem, scan);
}

// Copies of gradients (their strides kept), in one batched copy.
std::vector<torch::Tensor> copies_of(const std::vector<torch::Tensor>& grads) {
    at::NoGradGuard guard;
    std::vector<torch::Tensor> out;
    out.reserve(grads.size());
    for (const torch::Tensor& g : grads) out.push_back(at::empty_like(g));
    if (!out.empty()) at::_foreach_copy_(out, grads);
    return out;
}

// p.grad (+)= its slice of `flat`, parameter after parameter; one without a gradient gets a view of the flat tensor.
void add_flat_grads(const std::vector<torch::Tensor>& params, const torch::Tensor& flat) {
    at::NoGradGuard guard;
    int64_t o = 0;
    for (const torch::Tensor& p : params) {
        const int64_t n = p.numel();
        TORCH_CHECK(o + n <= flat.numel(), "add_flat_grads: parameters and gradients do not match");
        if (p.requires_grad()) {
            at::Tensor g = flat.narrow(0, o, n).view(p.sizes());
            if (g.scalar_type() != p.scalar_type()) g = g.to(p.scalar_type());
            at::Tensor& mine = const_cast<torch::Tensor&>(p).mutable_grad();
            mine = mine.defined() ? mine + g : g;
        }
        o += n;
    }
    TORCH_CHECK(o == flat.numel(), "add_flat_grads: parameters and gradients do not match");
}

// The meta-net's 33 weights from its parameters: detached, fp32, contiguous; an entry that is a list of them (one per head)
// becomes their stack, the experts' get their two or one dimensions.  Empty where an entry is neither: `kind` is the class of a
// parameter, and what derives from it may see more than a tensor's own operations.
std::vector<torch::Tensor> meta_weights(py::list entries, py::object kind, int64_t num_experts) {
    at::NoGradGuard guard;
    c10::AutoFwGradMode no_tangents(false);       // what is stacked below is not detached by itself
    auto parameter = [&](PyObject* o) { return o && (PyObject*)Py_TYPE(o) == kind.ptr() ? as_tensor(o) : nullptr; };
    const Py_ssize_t n = PyList_GET_SIZE(entries.ptr());
    std::vector<torch::Tensor> out;
    out.reserve(n);
    for (Py_ssize_t i = 0; i < n; i++) {
        PyObject* o = PyList_GET_ITEM(entries.ptr(), i);
        if (const at::Tensor* t = parameter(o)) {
            at::Tensor d = t->detach();
            if (d.scalar_type() != torch::kFloat32) d = d.to(torch::kFloat32);
            out.push_back(d.is_contiguous() ? d : d.contiguous());
            continue;
        }
        std::vector<at::Tensor> parts;
        for (Py_ssize_t k = 0; PyList_Check(o) && k < PyList_GET_SIZE(o); k++) {
            const at::Tensor* t = parameter(PyList_GET_ITEM(o, k));
            if (!t) return {};
            parts.push_back(t->scalar_type() == torch::kFloat32 ? *t : t->to(torch::kFloat32));
        }
        if (parts.empty()) return {};
        out.push_back(at::stack(parts));
    }
    if (n != SG2_NUM_WEIGHTS) return {};
    for (int k : {29, 31}) out[k] = out[k].reshape({num_experts, -1});
    out[32] = out[32].reshape({-1});
    return out;
}

// The random draws of an expert recycling event, in the order of the reference's loop
// (grokking_optimizers/mamba3_peer_metanet.py:453-488): per dead expert one N(0,1) draw for each of the four expert
// tensors into its row of `noise`, then a redraw of its key A row if every expert of that row is dead, then of its key B
// row.  A row is redrawn once per dead expert that shares it and only the last draw stays: the ones before are not
// drawn, the generator's offset moves past them (after one of them has shown by how much).
void recycle_draws(const std::vector<torch::Tensor>& noise, const std::vector<torch::Tensor>& keys_a, const std::vector<torch::Tensor>& keys_b,
                   const std::vector<int64_t>& dead, const std::vector<bool>& row_dead, const std::vector<bool>& col_dead, int64_t pk,
                   int64_t experts) {
    at::NoGradGuard guard;
    std::vector<std::vector<at::Tensor>> rows;
    for (const torch::Tensor& t : noise) rows.push_back(t.unbind(0));
    const bool skip = noise[0].is_cuda();
    at::Generator gen = at::globalContext().defaultGenerator(noise[0].device());
    uint64_t stride = 0;       // generator offset of one key row's draw
    auto redraw = [&](const std::vector<torch::Tensor>& keys, int64_t row, bool stays) {
        for (const torch::Tensor& k : keys) {
            if (skip && !stays && stride > 0) {
                gen.set_offset(gen.get_offset() + stride);
                continue;
            }
            const uint64_t before = skip ? gen.get_offset() : 0;
            at::Tensor r = k.select(0, row);
            if (stays) r.normal_().mul_(0.02);
            else at::empty_like(r).normal_();
            if (skip) stride = gen.get_offset() - before;
        }
    };
    for (size_t k = 0; k < dead.size(); k++) {
        const int64_t i = dead[k], a = i / pk, b = i % pk;
        for (auto& r : rows) r[k].normal_();
        if (row_dead[a]) redraw(keys_a, a, i == std::min(experts, (a + 1) * pk) - 1);
        if (col_dead[b]) redraw(keys_b, b, i + pk >= experts);
    }
}

constexpr int64_t RECYCLE_MAX_ROW = 65536;         // 256 values per CU

// Whether k_redraw_keys' draws are the framework's: the layout of a draw (how far it moves the generator's offset, which words
// of which counter an element takes) is no documented interface and may change with the framework or the device.  Rows of one
// value, of an odd length and of the largest one are drawn both ways from a generator of their own, once per device (a
// property of the two, not of any object); where they differ recycling takes recycle_draws.
bool draws_agree(const std::vector<torch::Tensor>& ours, const std::vector<torch::Tensor>& theirs) {
    for (size_t k = 0; k < ours.size(); k++) {
        const torch::Tensor d = (ours[k] - theirs[k]).abs().max();
        if (!(d.item<float>() < 1e-5f)) return false;       // deviations of 0.02: another layout is off by as much, another rounding of log, root and sine by 1e-6
    }
    return true;
}
bool generator_is_known(const torch::Device& device) {
    static std::mutex mutex;
    static std::map<int, bool> known;
    std::lock_guard<std::mutex> lock(mutex);
    const auto it = known.find(device.index());
    if (it != known.end()) return it->second;
    at::NoGradGuard guard;
    c10::DeviceGuard on(device);
    at::Generator shared = at::globalContext().defaultGenerator(device);
    at::Generator gen = [&] {
        std::lock_guard<std::mutex> held(shared.mutex());
        return shared.clone();
    }();
    gen.set_current_seed(0x9E3779B97F4A7C15ull);
    gen.set_offset(12);
    const auto opt = torch::TensorOptions().device(device).dtype(torch::kFloat32);
    std::vector<torch::Tensor> ours, theirs;
    std::vector<float*> rows;
    std::vector<int> lengths, draws;
    for (const int64_t n : {(int64_t)1, (int64_t)301, RECYCLE_MAX_ROW}) {
        lengths.push_back((int)n);
        draws.push_back((int)draws.size());
        ours.push_back(torch::empty({n}, opt));
        rows.push_back(ours.back().data_ptr<float>());
        theirs.push_back(torch::empty({n}, opt).normal_(0.0, 1.0, gen).mul_(0.02));
    }
    bool same = gen.get_offset() == 12 + 4 * lengths.size();
    if (same) {
        SgRecycle r = {};
        r.num_experts = 1;
        r.num_keys = (int)rows.size();
        r.key_rows = rows.data();
        r.key_lengths = lengths.data();
        r.key_draws = draws.data();
        r.seed = gen.current_seed();
        r.offset = 12;
        at::Tensor ws = at::empty({16 * (int64_t)rows.size()}, opt.dtype(at::kByte));
        check_status(sg_recycle_experts(&r, ws.data_ptr(), (size_t)ws.numel(), current_stream(ws)), "recycle_experts");
        same = draws_agree(ours, theirs);
    }
    known[device.index()] = same;
    return same;
}

// The same event for float32 parameters on the GPU: all draws in two launches.  False (nothing changed) where that is not
// what the tensors are, where a row is so long that its draw is not a block of the generator, or where the generator draws
// otherwise than the kernels.
bool recycle_experts(const std::vector<torch::Tensor>& experts, const std::vector<torch::Tensor>& keys_a, const std::vector<torch::Tensor>& keys_b,
                     const std::vector<int64_t>& dead, const std::vector<bool>& row_dead, const std::vector<bool>& col_dead, int64_t pk,
                     int64_t num_experts, int64_t top) {
    const torch::Tensor& first = experts.at(0);
    if (experts.size() != 4) return false;
    for (const auto* list : {&experts, &keys_a, &keys_b})
        for (const torch::Tensor& t : *list)
            if (!t.is_cuda() || t.device() != first.device() || t.scalar_type() != at::kFloat || !t.is_contiguous() || t.dim() < 1 || t.numel() == 0 ||
                t.numel() / t.size(0) > RECYCLE_MAX_ROW)
                return false;
    for (const torch::Tensor& t : experts)
        if (t.size(0) != num_experts) return false;
    for (const auto* list : {&keys_a, &keys_b})
        for (const torch::Tensor& t : *list)
            if (t.size(0) < pk) return false;
    if (!generator_is_known(first.device())) return false;
    c10::DeviceGuard device(first.device());
    std::vector<int> index, draw, key_lengths, key_draws;
    std::vector<float*> key_rows;
    int draws = 0;
    auto redraw = [&](const std::vector<torch::Tensor>& keys, int64_t row, bool stays) {
        for (const torch::Tensor& k : keys) {
            if (stays) {
                const int64_t n = k.numel() / k.size(0);
                key_rows.push_back(k.data_ptr<float>() + row * n);
                key_lengths.push_back((int)n);
                key_draws.push_back(draws);
            }
            draws++;
        }
    };
    for (const int64_t i : dead) {
        const int64_t a = i / pk, b = i % pk;
        index.push_back((int)i);
        draw.push_back(draws);
        draws += 4;
        if (row_dead.at(a)) redraw(keys_a, a, i == std::min(num_experts, (a + 1) * pk) - 1);
        if (col_dead.at(b)) redraw(keys_b, b, i + pk >= num_experts);
    }
    at::Generator gen = at::globalContext().defaultGenerator(first.device());
    SgRecycle r = {};
    {
        std::lock_guard<std::mutex> lock(gen.mutex());
        r.seed = gen.current_seed();
        r.offset = gen.get_offset();
        if (r.offset % 4 != 0) return false;
        gen.set_offset(r.offset + 4 * (uint64_t)draws);
    }
    for (int k = 0; k < 4; k++) {
        r.tensors[k] = experts[k].data_ptr<float>();
        r.row[k] = (int)(experts[k].numel() / num_experts);
    }
    r.num_experts = (int)num_experts;
    r.num_dead = (int)index.size();
    r.num_keys = (int)key_rows.size();
    r.top = (int)top;
    r.dead = index.data();
    r.draw = draw.data();
    r.key_rows = key_rows.data();
    r.key_lengths = key_lengths.data();
    r.key_draws = key_draws.data();
    const int64_t bytes = 16 * (int64_t)key_rows.size() + 8 * (int64_t)index.size();
    at::Tensor ws = at::empty({bytes}, first.options().dtype(at::kByte));
    check_status(sg_recycle_experts(&r, ws.data_ptr(), (size_t)bytes, current_stream(first)), "recycle_experts");
    return true;
}

// Whether a profiler record around a call could be seen: by a running profiler, by callbacks that an observer has added
// without one (execution traces, itt and nvtx ranges), or as an operator by a dispatch or function mode of this thread.
bool calls_are_observed() {
    return at::hasCallbacks() || torch::autograd::profiler::profilerEnabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           at::impl::torch_function_mode_enabled();
}

}  // namespace

void bind_group_steps(pybind11::module_& m) {
    m.def("calls_are_observed", &calls_are_observed);
    m.def("grokfast_group_step", &grokfast_group_step);
    m.def("lion_group_step", &lion_group_step);
    m.def("grokadamw_group_step", &grokadamw_group_step);
    m.def("adamw_group_step", &adamw_group_step);
    m.def("amplifier_on", &amplifier_on);
    m.def("neuralgrok_group_step", &neuralgrok_group_step);
    m.def("prodigy_group_step", &prodigy_group_step);
    m.def("muon_group_step", &muon_group_step);
    m.def("supergrok15_flat_step", &supergrok15_flat_step);
    m.def("supergrok11_flat_step", &supergrok11_flat_step);
    m.def("supergrok2_flat_step", &supergrok2_flat_step);
    py::class_<BilevelPass>(m, "BilevelPass");
    m.def("supergrok2_bilevel_begin", &supergrok2_bilevel_begin);
    m.def("supergrok2_bilevel_finish", &supergrok2_bilevel_finish);
    m.def("copies_of", &copies_of);
    m.def("add_flat_grads", &add_flat_grads);
    m.def("meta_weights", &meta_weights);
    m.def("recycle_draws", &recycle_draws);
    m.def("recycle_experts", &recycle_experts);
    m.def("draws_agree", &draws_agree);
}

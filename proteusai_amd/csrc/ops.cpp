// The operators' host path in C++: allocations, launches and autograd nodes of geometric attention and of the two wavefunction embeddings for ordinary calls.
//
// Every function here takes a call only if it is the plain one -- ordinary tensors of the kernels' own types and layouts on the current GPU, and nothing that looks on (functional
// transforms, forward-mode differentiation, dispatch modes, tracing) -- and answers None otherwise: the Python functions, which convert, check and raise, do the
// rest, and the backward of a node hands whatever is not plain (gradients without memory of their own, saved tensors that hooks gave back in another form) to them, too.
// Us of a forward and backward that the host bounds, Python / this: attention of 64 tokens 86 to 170 / 46 to 80 (the higher figures are processes whose autograd thread
// waits longer for the interpreter's lock, which the backward no longer takes), with the spreads checked 110 to 193 / 56, embedding of 2 x 512 70 to 131 / 48; a forward alone 11.5 / 7.1 and
// 22.6 / 18.5 (the GPU's time).
#include <torch/extension.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include "proteus_hip.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

// ---- which calls ----

// Does nothing look on that expects torch operators?
bool unobserved()
{
    return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing();
}

// A tensor with memory of its own on the current GPU that carries no tangent.
bool plain(const Tensor& t)
{
    if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda()) return false;
    const auto keys = t.unsafeGetTensorImpl()->key_set();
    return !keys.has(c10::DispatchKey::Python) && !keys.has(c10::DispatchKey::FuncTorchBatched) && !keys.has(c10::DispatchKey::FuncTorchGradWrapper)
           && !keys.has(c10::DispatchKey::Functionalize) && !keys.has(c10::DispatchKey::ZeroTensor) && !keys.has(c10::DispatchKey::Negative)
           && t.has_storage() && !t._fw_grad(0).defined();
}

// The tensor behind a Python object that is exactly a Tensor or Parameter and plain, on device `dev` (any, the current one, where that is negative).
bool get(const py::object& o, Tensor& t, const int dev = -1)
{
    if (!THPVariable_CheckExact(o.ptr())) return false;
    t = THPVariable_Unpack(o.ptr());
    return plain(t) && (dev < 0 || t.get_device() == dev);
}

bool f32(const Tensor& t) { return t.scalar_type() == at::kFloat && t.is_contiguous(); }
const float* floats(const Tensor& t) { return static_cast<const float*>(t.const_data_ptr()); }
float* out_floats(const Tensor& t) { return static_cast<float*>(t.mutable_data_ptr()); }
const uint16_t* halves(const Tensor& t) { return static_cast<const uint16_t*>(t.const_data_ptr()); }
const uint8_t* bytes(const Tensor& t) { return t.defined() ? static_cast<const uint8_t*>(t.const_data_ptr()) : nullptr; }
bool off(const Tensor& t, const uintptr_t by) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & (by - 1)) != 0; }

// An optional padding mask [Z, N]: None, or a dense bool tensor.
bool get_mask(const py::object& o, Tensor& m, const int dev, const int64_t Z, const int64_t N)
{
    if (o.is_none()) return true;
    return get(o, m, dev) && m.scalar_type() == at::kBool && m.is_contiguous() && m.dim() == 2 && m.size(0) == Z && m.size(1) == N;
}

bool current(const int dev)
{
    int now = -1;
    return hipGetDevice(&now) == hipSuccess && now == dev;
}

void* stream_of(const int dev) { return c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream(); }

// What the library does not take, or could not launch, goes the general way, which says what is wrong with it (as a ValueError or a ProteusError).
struct Refused {};
void launched(const int rc) { if (rc != 0) throw Refused(); }

at::TensorOptions on(const Tensor& t, const at::ScalarType type) { return t.options().dtype(type).requires_grad(false); }

// ---- geometric attention ----

// Can the kernels read or write this [Z,H,N,d] tensor in place?  (Rows of d contiguous elements on multiples of 16 bytes, no negative or overlapping strides.)
bool rows_ok(const Tensor& t, const int64_t itemsize)
{
    if (off(t, 16)) return false;
    if (t.is_contiguous()) return true;
    const int64_t per16 = 16 / itemsize;
    if (t.stride(3) != 1 || t.stride(2) < t.size(3) || t.size(2) * t.stride(2) * itemsize >= (1LL << 31)) return false;
    for (int i = 0; i < 3; ++i) if (t.stride(i) < 0 || t.stride(i) % per16) return false;
    return (t.size(0) == 1 || t.stride(0) > 0) && (t.size(1) == 1 || t.stride(1) > 0);
}

struct Strides {
    int64_t v[21];
    bool dense = true;
    int n = 0;
    void add(const Tensor& t) { for (int i = 0; i < 3; ++i) v[n++] = t.stride(i); dense = dense && t.is_contiguous(); }
    const int64_t* get() const { return dense ? nullptr : v; }
};

struct Logits { bool legacy, f16; double min_rbf, max_rbf; };

std::pair<Tensor, Tensor> attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& coords, const Tensor& sigma, const Tensor& betas, const Tensor& mask,
                                            const Logits& how, const bool token_major)
{
    const int64_t Z = q.size(0), H = q.size(1), N = q.size(2), d = q.size(3);
    const auto opt = on(q, at::kFloat);
    const Tensor O = token_major ? at::empty({Z, N, H, d}, opt).permute({0, 2, 1, 3}) : at::empty({Z, H, N, d}, opt);
    const Tensor L = at::empty({Z, H, N}, opt);
    Strides st;
    for (const Tensor* t : {&q, &k, &v, &O}) st.add(*t);
    void* const stream = stream_of(q.get_device());
    if (!how.legacy) {
        const size_t need = proteus_geo_attn_fwd_workspace_bytes(Z, H, N, d, 0);
        Tensor ws;
        if (need) ws = at::empty({static_cast<int64_t>(need)}, on(q, at::kByte));
        launched(proteus_geo_attn_fwd_ws(halves(q), halves(k), halves(v), st.get(), floats(coords), floats(sigma), bytes(mask), out_floats(O), out_floats(L),
                                         need ? ws.mutable_data_ptr() : nullptr, need, Z, H, N, d, 0, stream));
    } else {
        // (contiguous tensors may have any stride along a dimension of size one, which the strided entry point would hold against them)
        const int type = how.f16 ? PROTEUS_OPERAND_F16 : PROTEUS_OPERAND_BF16;
        launched(st.get() ? proteus_geo_attn_legacy_fwd_strided(halves(q), halves(k), halves(v), st.get(), floats(coords), floats(sigma), floats(betas), bytes(mask), out_floats(O), out_floats(L),
                                                                Z, H, N, d, how.min_rbf, how.max_rbf, type, 0, stream)
                          : proteus_geo_attn_legacy_fwd(halves(q), halves(k), halves(v), floats(coords), floats(sigma), floats(betas), bytes(mask), out_floats(O), out_floats(L),
                                                        Z, H, N, d, how.min_rbf, how.max_rbf, type, 0, stream));
    }
    return {O, L};
}

PyObject* g_attention_backward = nullptr;        // the Python function (set once, when the module is set up)

// What is not plain: gradients and saved tensors as the Python function takes them.
variable_list attention_backward_general(const variable_list& s, const Tensor& dO, const Logits& how)
{
    py::gil_scoped_acquire gil;
    auto opt = [](const Tensor& t) -> py::object { return t.defined() ? py::cast(t) : py::none(); };
    const py::object got = py::reinterpret_borrow<py::object>(g_attention_backward)(s[0], s[1], s[2], s[3], s[4], dO, s[5], s[6], opt(s[8]), opt(s[7]), how.min_rbf, how.max_rbf, how.f16);
    variable_list out;
    for (const auto& o : py::reinterpret_borrow<py::tuple>(got)) out.push_back(o.is_none() ? Tensor() : o.cast<Tensor>());
    return out;                                  // dQ, dK, dV, d_sigma, d_betas
}

variable_list attention_backward_plain(const variable_list& s, const Tensor& dO, const Logits& how)
{
    const Tensor &q = s[0], &k = s[1], &v = s[2], &O = s[3], &L = s[4], &coords = s[5], &sigma = s[6], &betas = s[7], &mask = s[8];
    const auto op = how.f16 ? at::kHalf : at::kBFloat16;
    const auto type = dO.defined() ? dO.scalar_type() : at::kByte;
    bool ok = unobserved() && (type == at::kFloat || type == at::kBFloat16 || type == at::kHalf) && plain(dO) && current(dO.get_device()) && O.dim() == 4 && O.sizes() == dO.sizes();
    for (const Tensor* t : {&q, &k, &v}) ok = ok && plain(*t) && t->scalar_type() == op && t->sizes() == O.sizes() && rows_ok(*t, 2);
    for (const Tensor* t : {&L, &coords, &sigma}) ok = ok && plain(*t) && f32(*t);
    ok = ok && plain(O) && O.scalar_type() == at::kFloat;
    if (!ok) return attention_backward_general(s, dO, how);
    const int64_t Z = O.size(0), H = O.size(1), N = O.size(2), d = O.size(3);
    ok = L.numel() == Z * H * N && coords.numel() == Z * N * 3 && sigma.numel() == H;
    for (const Tensor* t : {&q, &k, &v, &O, &L, &coords, &sigma}) ok = ok && t->get_device() == dO.get_device();
    if (betas.defined()) ok = ok && plain(betas) && f32(betas) && betas.numel() == H && betas.get_device() == dO.get_device();
    if (mask.defined())  ok = ok && plain(mask) && mask.scalar_type() == at::kBool && mask.is_contiguous() && mask.numel() == Z * N && mask.get_device() == dO.get_device();
    ok = ok && !off(O, 16) && !off(dO, 4 * dO.element_size());
    if (!(O.is_contiguous() && dO.is_contiguous()))
        for (const Tensor* t : {&O, &dO}) {
            ok = ok && t->stride(3) == 1 && t->stride(2) >= d;
            for (int i = 0; i < 3; ++i) ok = ok && t->stride(i) % 4 == 0;
        }
    if (!ok) return attention_backward_general(s, dO, how);
    Tensor cast = dO;
    if (type != op) cast = at::empty_like(dO, on(dO, op));
    if (!rows_ok(cast, 2)) return attention_backward_general(s, dO, how);

    const auto opt = on(O, at::kFloat);
    const Tensor D = at::empty({Z, H, N}, opt), d_sigma = at::empty({H}, opt);
    const Tensor d_beta = betas.defined() ? at::empty({H}, opt) : Tensor();
    float* const to_beta = betas.defined() ? out_floats(d_beta) : nullptr;
    const int operand = how.f16 ? PROTEUS_OPERAND_F16 : PROTEUS_OPERAND_BF16;
    void* const stream = stream_of(O.get_device());
    Strides prep;
    for (const Tensor* t : {&O, &dO, static_cast<const Tensor*>(&cast)}) prep.add(*t);
    launched(proteus_geo_attn_prepare_bwd(floats(O), dO.const_data_ptr(), prep.get(), out_floats(D), type != op ? static_cast<uint16_t*>(cast.mutable_data_ptr()) : nullptr, out_floats(d_sigma),
                                          to_beta, Z, H, N, d, type == at::kFloat ? PROTEUS_DTYPE_F32 : type == at::kHalf ? PROTEUS_DTYPE_F16 : PROTEUS_DTYPE_BF16, operand, stream));
    // gradients in the memory order of their operands (dense) and in their type
    auto like = [&](const Tensor& t) {
        const Tensor g = at::empty_like(t, on(t, op));
        return rows_ok(g, 2) ? g : at::empty({Z, H, N, d}, on(t, op));
    };
    const Tensor dq = like(q), dk = like(k), dv = like(v);
    Strides st;
    for (const Tensor* t : {&q, &k, &v, static_cast<const Tensor*>(&cast), &dq, &dk, &dv}) st.add(*t);
    launched(proteus_geo_attn_bwd_typed(halves(q), halves(k), halves(v), halves(cast), st.get(), floats(coords), floats(sigma), betas.defined() ? floats(betas) : nullptr, bytes(mask),
                                        floats(L), floats(D), dq.mutable_data_ptr(), dk.mutable_data_ptr(), dv.mutable_data_ptr(), out_floats(d_sigma), to_beta, Z, H, N, d,
                                        how.legacy ? how.min_rbf : 0.0, how.legacy ? how.max_rbf : 1.0, operand, PROTEUS_GRAD_OPERAND, stream));
    return {dq, dk, dv, d_sigma, d_beta};
}

variable_list attention_backward(const variable_list& s, const Tensor& dO, const Logits& how)
{
    try {
        return attention_backward_plain(s, dO, how);
    } catch (const Refused&) {
        return attention_backward_general(s, dO, how);
    }
}

struct Attention : torch::autograd::Function<Attention> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& coords, const Tensor& spreads,
                          const std::optional<Tensor>& betas, const std::optional<Tensor>& mask, bool legacy, bool f16, double min_rbf, double max_rbf, bool token_major)
    {
        const Tensor b = betas.value_or(Tensor()), m = mask.value_or(Tensor());
        const auto [O, L] = attention_forward(q, k, v, coords, spreads, b, m, Logits{legacy, f16, min_rbf, max_rbf}, token_major);
        ctx->save_for_backward({q, k, v, O, L, coords, spreads, b, m});
        ctx->saved_data["legacy"] = legacy; ctx->saved_data["f16"] = f16;
        ctx->saved_data["min"] = min_rbf; ctx->saved_data["max"] = max_rbf;
        return O;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const Logits how{ctx->saved_data["legacy"].toBool(), ctx->saved_data["f16"].toBool(), ctx->saved_data["min"].toDouble(), ctx->saved_data["max"].toDouble()};
        const variable_list g = attention_backward(ctx->get_saved_variables(), grads[0], how);
        return {g[0], g[1], g[2], Tensor(), g[3], g[4], Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// The spreads' values on their way to the host while the kernels that read them are launched: a call that waited for them first left the GPU without work for
// as long as the host then takes to launch.
struct Arriving {
    Tensor host;
    hipEvent_t done = nullptr;
    Arriving(const Tensor& t, hipStream_t stream)
    {
        host = at::empty({t.numel()}, at::TensorOptions().dtype(at::kFloat).device(at::kCPU).pinned_memory(true));
        if (hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess) { done = nullptr; return; }
        if (hipMemcpyAsync(host.mutable_data_ptr(), t.const_data_ptr(), t.numel() * 4, hipMemcpyDeviceToHost, stream) != hipSuccess || hipEventRecord(done, stream) != hipSuccess) {
            (void)hipStreamSynchronize(stream);
            (void)hipEventDestroy(done);
            done = nullptr;
        }
    }
    ~Arriving() { if (done) { (void)hipEventSynchronize(done); (void)hipEventDestroy(done); } }          // (the memory is written until then)
    // Once they are there: are all of them positive numbers?
    bool positive()
    {
        if (!done || hipEventSynchronize(done) != hipSuccess) return false;
        const float* v = floats(host);
        for (int64_t i = 0; i < host.numel(); ++i) if (!(v[i] > 0.0f)) return false;
        return true;
    }
};

// geometric_attn(...) with O in fp32, or None.
py::object attention(const py::object& Q, const py::object& K, const py::object& V, const py::object& coords_, const py::object& spreads_, const py::object& betas_, const py::object& mask_,
                     const double min_rbf, const double max_rbf, const bool check, const bool token_major, const bool f16)
{
    Tensor q, k, v, coords, spreads, betas, mask;
    if (!unobserved() || !get(Q, q) || q.dim() != 4) return py::none();
    const int dev = q.get_device();
    const int64_t Z = q.size(0), H = q.size(1), N = q.size(2), d = q.size(3);
    const auto op = f16 ? at::kHalf : at::kBFloat16;
    const bool legacy = !betas_.is_none();
    if ((f16 && !legacy) || !current(dev) || !get(K, k, dev) || !get(V, v, dev) || !get(coords_, coords, dev) || !get(spreads_, spreads, dev) || !get_mask(mask_, mask, dev, Z, N)
        || (legacy && !get(betas_, betas, dev))) return py::none();
    for (const Tensor* t : {&q, &k, &v}) if (t->scalar_type() != op || t->sizes() != q.sizes() || !rows_ok(*t, 2)) return py::none();
    if (Z <= 0 || H <= 0 || N <= 0 || (d != 32 && d != 64 && d != 128) || N > PROTEUS_ATTN_MAX_N || Z * H > 65535
        || !f32(coords) || coords.dim() != 3 || coords.size(0) != Z || coords.size(1) != N || coords.size(2) != 3
        || !f32(spreads) || spreads.dim() != 1 || spreads.size(0) != H || (legacy && (!f32(betas) || betas.dim() != 1 || betas.size(0) != H || !(max_rbf > min_rbf)))
        || N * H * d * 4 >= (1LL << 31)) return py::none();
    const hipStream_t stream = static_cast<hipStream_t>(stream_of(dev));
    std::optional<Arriving> arriving;
    if (check) {
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) return py::none();
        arriving.emplace(spreads, stream);
    }
    const bool recording = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad() || spreads.requires_grad() || (legacy && betas.requires_grad()));
    Tensor O;
    bool good = true;
    try {
        py::gil_scoped_release no_gil;
        const std::optional<Tensor> b = legacy ? std::optional<Tensor>(betas) : std::nullopt, m = mask.defined() ? std::optional<Tensor>(mask) : std::nullopt;
        if (recording) O = Attention::apply(q, k, v, coords, spreads, b, m, legacy, f16, min_rbf, max_rbf, token_major);
        else {
            at::NoGradGuard no_grad;
            O = attention_forward(q, k, v, coords, spreads, betas, mask, Logits{legacy, f16, min_rbf, max_rbf}, token_major).first;
        }
        if (arriving) good = arriving->positive();
    } catch (const Refused&) {
        return py::none();
    }
    return good ? py::cast(O) : py::none();                   // (what is wrong with the spreads is said by the general path)
}

// ---- wavefunction embedding ----

PyObject* g_embedding_backward = nullptr;
PyObject* g_aniso_backward = nullptr;

// A gradient, and what the forward kept for it, that the kernels may read.
bool backward_ok(const Tensor& dO, const variable_list& kept, const int64_t per_gradient)
{
    if (!unobserved() || !dO.defined() || !plain(dO) || !f32(dO) || dO.dim() != 3 || off(dO, 8) || !current(dO.get_device())) return false;
    for (const Tensor& t : kept)
        if (t.defined() && !(plain(t) && f32(t) && t.get_device() == dO.get_device() && t.numel() * per_gradient == dO.numel() && !off(t, 8))) return false;
    return true;
}

Tensor bwd_workspace(const Tensor& dO, const int64_t K)
{
    return at::empty({static_cast<int64_t>(proteus_we_bwd_workspace_bytes(dO.size(0), dO.size(1), K))}, on(dO, at::kByte));
}

std::array<Tensor, 3> embedding_forward(const Tensor& coords, const Tensor& wn, const Tensor& mask, const bool sums)
{
    const int64_t Z = coords.size(0), N = coords.size(1), K = wn.size(0);
    const auto opt = on(coords, at::kFloat);
    const Tensor out = at::empty({Z, N, 2 * K}, opt);
    const Tensor cs = sums ? at::empty({Z, N, K}, opt) : Tensor(), sn = sums ? at::empty({Z, N, K}, opt) : Tensor();
    const size_t need = proteus_we_fwd_workspace_bytes(Z, N, K, 0);
    Tensor ws;
    if (need) ws = at::empty({static_cast<int64_t>(need)}, on(coords, at::kByte));
    launched(proteus_we_fwd_ws(floats(coords), PROTEUS_COORDS_AOS, floats(wn), bytes(mask), out_floats(out), sums ? out_floats(cs) : nullptr, sums ? out_floats(sn) : nullptr,
                               need ? ws.mutable_data_ptr() : nullptr, need, Z, N, K, 0, stream_of(coords.get_device())));
    return {out, cs, sn};
}

struct Embedding : torch::autograd::Function<Embedding> {
    static Tensor forward(AutogradContext* ctx, const Tensor& coords, const Tensor& wn, const std::optional<Tensor>& mask)
    {
        const auto [out, cs, sn] = embedding_forward(coords, wn, mask.value_or(Tensor()), true);
        ctx->save_for_backward({cs, sn});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list s = ctx->get_saved_variables();
        const Tensor& dO = grads[0];
        if (backward_ok(dO, s, 2)) try {
            return {Tensor(), reduced(dO, s), Tensor()};
        } catch (const Refused&) {}
        py::gil_scoped_acquire gil;
        return {Tensor(), py::reinterpret_borrow<py::object>(g_embedding_backward)(dO, s[0], s[1]).cast<Tensor>(), Tensor()};
    }
    static Tensor reduced(const Tensor& dO, const variable_list& s)
    {
        const int64_t K = dO.size(2) / 2;
        const Tensor ws = bwd_workspace(dO, K), dk = at::empty({K}, on(dO, at::kFloat));
        launched(proteus_we_bwd(floats(dO), floats(s[0]), floats(s[1]), out_floats(dk), out_floats(ws), ws.numel(), dO.size(0), dO.size(1), K, stream_of(dO.get_device())));
        return dk;
    }
};

std::array<Tensor, 3> aniso_forward(const Tensor& a, const Tensor& b, const Tensor& cb, const Tensor& wn, const Tensor& mask, const bool partials)
{
    const int64_t Z = a.size(0), N = a.size(1), K = wn.size(0);
    const auto opt = on(a, at::kFloat);
    const Tensor out = at::empty({Z, N, 2 * K}, opt);
    const Tensor d_cb = partials ? at::empty({Z, N, 2 * K}, opt) : Tensor(), d_k = partials ? at::empty({Z, N, 2 * K}, opt) : Tensor();
    const size_t need = proteus_we_aniso_fwd_workspace_bytes(Z, N, K, partials, mask.defined(), 0);
    Tensor ws;
    if (need) ws = at::empty({static_cast<int64_t>(need)}, on(a, at::kByte));
    launched(proteus_we_aniso_fwd_ws(floats(a), floats(b), PROTEUS_COORDS_AOS, floats(cb), floats(wn), bytes(mask), out_floats(out), partials ? out_floats(d_cb) : nullptr,
                                     partials ? out_floats(d_k) : nullptr, need ? ws.mutable_data_ptr() : nullptr, need, Z, N, K, 0, stream_of(a.get_device())));
    return {out, d_cb, d_k};
}

struct Aniso : torch::autograd::Function<Aniso> {
    static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b, const Tensor& cb, const Tensor& wn, const std::optional<Tensor>& mask)
    {
        const auto [out, d_cb, d_k] = aniso_forward(a, b, cb, wn, mask.value_or(Tensor()), true);
        ctx->save_for_backward({d_cb, d_k});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        variable_list s = ctx->get_saved_variables();
        const Tensor& dO = grads[0];
        for (int i = 0; i < 2; ++i) if (!ctx->needs_input_grad(2 + i)) s[i] = Tensor();
        if (!s[0].defined() && !s[1].defined()) return {Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
        if (backward_ok(dO, s, 1)) try {
            return reduced(dO, s);
        } catch (const Refused&) {}
        py::gil_scoped_acquire gil;
        auto opt = [](const Tensor& t) -> py::object { return t.defined() ? py::cast(t) : py::none(); };
        const py::tuple got = py::reinterpret_borrow<py::object>(g_aniso_backward)(dO, opt(s[0]), opt(s[1]));
        auto back = [&](const int i) { const py::object o = got[i]; return o.is_none() ? Tensor() : o.cast<Tensor>(); };
        return {Tensor(), Tensor(), back(0), back(1), Tensor()};
    }
    static variable_list reduced(const Tensor& dO, const variable_list& s)
    {
        const int64_t K = dO.size(2) / 2;
        const Tensor ws = bwd_workspace(dO, K);
        Tensor g[2];
        for (int i = 0; i < 2; ++i) if (s[i].defined()) g[i] = at::empty({K}, on(dO, at::kFloat));
        launched(proteus_we_aniso_bwd(floats(dO), s[0].defined() ? floats(s[0]) : nullptr, s[1].defined() ? floats(s[1]) : nullptr, g[0].defined() ? out_floats(g[0]) : nullptr,
                                      g[1].defined() ? out_floats(g[1]) : nullptr, out_floats(ws), ws.numel(), dO.size(0), dO.size(1), K, stream_of(dO.get_device())));
        return {Tensor(), Tensor(), g[0], g[1], Tensor()};
    }
};

bool sizes_ok(const Tensor& coords, const Tensor& wn)
{
    return f32(coords) && coords.dim() == 3 && coords.size(2) == 3 && f32(wn) && wn.dim() == 1 && coords.size(0) > 0 && coords.size(0) <= 65535 && coords.size(1) > 0
           && coords.size(1) <= PROTEUS_WE_MAX_N && wn.size(0) > 0 && wn.size(0) <= PROTEUS_WE_MAX_K;
}

// wf_embedding(coords, wavenumbers, mask=mask), or None.
py::object embedding(const py::object& coords_, const py::object& wn_, const py::object& mask_)
{
    Tensor coords, wn, mask;
    if (!unobserved() || !get(coords_, coords) || !current(coords.get_device()) || !get(wn_, wn, coords.get_device()) || !sizes_ok(coords, wn)
        || !get_mask(mask_, mask, coords.get_device(), coords.size(0), coords.size(1)) || coords.requires_grad()) return py::none();
    Tensor out;
    try {
        py::gil_scoped_release no_gil;
        if (at::GradMode::is_enabled() && wn.requires_grad()) out = Embedding::apply(coords, wn, mask.defined() ? std::optional<Tensor>(mask) : std::nullopt);
        else { at::NoGradGuard no_grad; out = embedding_forward(coords, wn, mask, false)[0]; }
    } catch (const Refused&) {
        return py::none();
    }
    return py::cast(out);
}

// wf_embedding_learnCB(a, b, cb, wavenumbers, mask), or None.
py::object aniso(const py::object& a_, const py::object& b_, const py::object& cb_, const py::object& wn_, const py::object& mask_)
{
    Tensor a, b, cb, wn, mask;
    if (!unobserved() || !get(a_, a) || !current(a.get_device())) return py::none();
    const int dev = a.get_device();
    if (!get(b_, b, dev) || !get(cb_, cb, dev) || !get(wn_, wn, dev) || !sizes_ok(a, wn) || !f32(b) || b.sizes() != a.sizes() || !f32(cb) || cb.sizes() != wn.sizes()
        || !get_mask(mask_, mask, dev, a.size(0), a.size(1)) || a.requires_grad() || b.requires_grad()) return py::none();
    Tensor out;
    try {
        py::gil_scoped_release no_gil;
        if (at::GradMode::is_enabled() && (cb.requires_grad() || wn.requires_grad())) out = Aniso::apply(a, b, cb, wn, mask.defined() ? std::optional<Tensor>(mask) : std::nullopt);
        else { at::NoGradGuard no_grad; out = aniso_forward(a, b, cb, wn, mask, false)[0]; }
    } catch (const Refused&) {
        return py::none();
    }
    return py::cast(out);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("version", [] { return proteus_version(); });
    m.def("attention", &attention);
    m.def("embedding", &embedding);
    m.def("aniso", &aniso);
    // the general backward functions (kept for as long as the process lives)
    m.def("set_general", [](py::object attention_bwd, py::object embedding_bwd, py::object aniso_bwd) {
        g_attention_backward = attention_bwd.release().ptr();
        g_embedding_backward = embedding_bwd.release().ptr();
        g_aniso_backward = aniso_bwd.release().ptr();
    });
}

// Host side of the quantized layers as one native extension: the autograd functions of the Quartet linear, of the two
// layers whose producer is fused into them (RMSNorm, SwiGLU), of the rotary split and of the quantizer modules.  Every
// kernel is launched through the C ABI of libquartet_hip.so; PyTorch allocates, provides the stream and the graph.
//
// Why native: a training step of one layer is five to nine launches.  Driven from Python (autograd.Function, ctypes calls
// with thirty arguments, a dozen small helper calls) it took 220-250 us of host time whatever its size, so every layer
// whose kernels run shorter than that was bound by the interpreter.  Here the same step is a handful of allocations and
// the launches themselves.  The one thing that stays in Python is the drawing of random numbers: sign flips come from
// torch's host generator and seeds from the `random` module, in the order e, W^T, e^T, x^T, through one callback.
#include <torch/extension.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "../../include/quartet_hip.h"

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
using at::Tensor;
using std::optional;

PyObject* g_error_class = nullptr;   // quartet_amd._lib.QuartetHipError
PyObject* g_draw = nullptr;          // quartet_amd.linear._gradient_draws
PyObject* g_error_draw = nullptr;    // quartet_amd.linear._error_draws

// ---- errors: raised as Python exceptions, also from the autograd engine's threads --------------------------------
[[noreturn]] void raise(PyObject* type, const std::string& message) {
    py::gil_scoped_acquire gil;
    PyErr_SetString(type, message.c_str());
    python_error e;
    e.persist();
    throw e;
}
void check(int rc, const char* what) {
    if (rc != 0) raise(g_error_class, std::string(what) + " failed (rc=" + std::to_string(rc) + "): " + qm_last_error());
}
template <typename... Ts>
void require_cuda(const Ts&... tensors) {
    if (!(... && (!tensors.defined() || tensors.is_cuda())))
        raise(g_error_class, "quartet_amd kernels need tensors on the GPU (no CPU path exists)");
}
int dtype_code(at::ScalarType t) {
    if (t == at::kBFloat16) return QM_BF16;
    if (t == at::kFloat) return QM_F32;
    raise(PyExc_TypeError, std::string("quartet_amd kernels take bfloat16 or float32 tensors, got ") + c10::toString(t));
}
// entry points called from Python: hand a python_error over to the interpreter
template <typename F>
auto from_python(F&& f) {
    try {
        return f();
    } catch (python_error& e) {
        e.restore();
        throw py::error_already_set();
    }
}

// ---- small helpers ------------------------------------------------------------------------------------------------
bool autocast_bf16() { return at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) == at::kBFloat16; }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
Tensor bytes(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }
Tensor rows_of(const Tensor& t, int64_t cols) { return t.reshape({-1, cols}).contiguous(); }
const void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
Tensor or_none(const optional<Tensor>& t) { return t ? *t : Tensor(); }

// the accumulated column signs of a rotation: a Python int of hadamard_dim bits, or None
struct Signs {
    uint32_t w[4] = {0, 0, 0, 0};
    const uint32_t* data() const { return (w[0] | w[1] | w[2] | w[3]) ? w : nullptr; }
};
Signs signs_of(py::handle bits) {
    Signs s;
    if (bits.is_none()) return s;
    int overflow = 0;
    const long long low = PyLong_AsLongLongAndOverflow(bits.ptr(), &overflow);
    if (low == -1 && PyErr_Occurred()) throw py::error_already_set();
    if (!overflow) {
        s.w[0] = (uint32_t)low;
        s.w[1] = (uint32_t)((unsigned long long)low >> 32);
        return s;
    }
    py::object rest = py::reinterpret_borrow<py::object>(bits);
    const py::int_ shift(32), mask(0xffffffffu);
    for (int i = 0; i < 4; ++i) {
        s.w[i] = (rest & mask).cast<uint32_t>();
        rest = rest >> shift;
    }
    return s;
}

// An object of the interpreter kept by a graph node, which may be released by a thread that does not hold the GIL.
struct PyHandle {
    PyObject* p = nullptr;
    explicit PyHandle(py::handle h) : p(h.ptr()) { Py_XINCREF(p); }
    PyHandle(const PyHandle&) = delete;
    PyHandle& operator=(const PyHandle&) = delete;
    ~PyHandle() {
        if (p && Py_IsInitialized()) {
            py::gil_scoped_acquire gil;
            Py_DECREF(p);
        }
    }
};

// ---- the products of one layer --------------------------------------------------------------------------------------
// What the layer is configured to do and what its backward pass needs besides the packed operands.
struct Layer : torch::CustomClassHolder {
    PyHandle g_q;              // the gradient quantizer (sign flips and seeds are drawn from it in backward)
    int a_hd, w_hd, g_hd;
    Signs a_signs, w_signs;
    Tensor x_dense, w_dense;   // dense rotations of the forward quantizers (rerotate="O32"), or undefined
    int64_t T = 0, I = 0, O = 0;
    int layout = QM_LAYOUT_ROWMAJOR;
    bool seed_base_ok = false;
    bool error_only = false;   // scheme "Q(E)W_Q(Et)X": the gradient products take the packed operands as they are
    at::ScalarType x_dtype{}, w_dtype{};
    std::vector<int64_t> x_shape;
    explicit Layer(py::handle q) : g_q(q) {}
};
using LayerPtr = c10::intrusive_ptr<Layer>;

LayerPtr make_layer(int a_hd, py::handle a_signs, int w_hd, py::handle w_signs, int g_hd, py::handle g_q, const optional<Tensor>& x_dense,
                    const optional<Tensor>& w_dense) {
    auto l = c10::make_intrusive<Layer>(g_q);
    l->a_hd = a_hd; l->w_hd = w_hd; l->g_hd = g_hd;
    l->a_signs = signs_of(a_signs); l->w_signs = signs_of(w_signs);
    l->x_dense = or_none(x_dense); l->w_dense = or_none(w_dense);
    return l;
}

// contractions from here on are not the tile kernels' (csrc/gemm_tile.hip): 32-bit offsets inside a tile.  The packed-weight key
// of quartet_amd.linear holds which side of it a call's tokens are on.
constexpr int64_t kLongContraction = 1 << 23;

void set_extents(Layer& l, int64_t T, const Tensor& weight) {
    l.T = T; l.I = weight.size(1); l.O = weight.size(0);
    l.w_dtype = weight.scalar_type();
    // Tiled code bytes (16 rows x 128 elements contiguous, extents padded with zeros).  Row-major where the padding is not
    // available: rows of y that are not whole 16-byte pieces, and dense forward rotations off the multiples of 128; and where
    // an extent is too long a contraction for the tile kernels and the others too ragged or short for the 256 x 256 one.
    const bool dense = l.x_dense.defined() || l.w_dense.defined();
    const bool classic = l.T % 128 == 0 && l.I % 128 == 0 && l.O % 128 == 0;
    const bool large = classic && l.T >= 256 && l.I >= 256 && l.O >= 256;
    l.layout = l.O % 8 || (dense && !classic) || (std::max({l.T, l.I, l.O}) >= kLongContraction && !large) ? QM_LAYOUT_ROWMAJOR : QM_LAYOUT_PADDED;
    // the extents for which a device seed base is promised (set_device_seed_base)
    l.seed_base_ok = large && l.a_hd == 32 && l.w_hd == 32 && l.g_hd == 32;
}

Tensor packed_buffer(int64_t rows, int64_t cols, const Tensor& like) { return bytes((int64_t)qm_packed_operand_bytes(rows, cols), like); }
Tensor mask_bits(const Tensor& packed, int64_t rows, int64_t cols) {
    size_t off[3];
    check(qm_packed_operand_offsets(rows, cols, off), "qm_packed_operand_offsets");
    return packed.narrow(0, (int64_t)off[2], rows * cols / 8).view({rows, cols / 8});
}

// Quest RTN + clip mask under a dense 32 x 32 rotation, written into a fresh packed-operand buffer
Tensor quantize_dense_into_packed(const Tensor& x2, const Tensor& dense, int layout) {
    const int64_t rows = x2.size(0), cols = x2.size(1);
    // the matrix cast to the quantized tensor's dtype, as the quantizer modules cast it; fp32 storage for the kernel
    const Tensor m = dense.to(x2.device()).to(x2.scalar_type()).to(at::kFloat).contiguous();
    if (m.dim() != 2 || m.size(0) != 32 || m.size(1) != 32) raise(g_error_class, "a dense rotation must be 32 x 32");
    Tensor packed = packed_buffer(rows, cols, x2);
    size_t off[3];
    check(qm_packed_operand_offsets(rows, cols, off), "qm_packed_operand_offsets");
    uint8_t* base = packed.data_ptr<uint8_t>();
    check(qm_quantize_mxfp4_dense(x2.data_ptr(), dtype_code(x2.scalar_type()), rows, cols, m.data_ptr<float>(), QM_QUEST_RTN, 0, 0,
                                  base + off[0], base + off[1], base + off[2], nullptr, layout == QM_LAYOUT_PADDED ? QM_LAYOUT_TILED : layout, stream_of(x2)),
          "qm_quantize_mxfp4_dense");
    return packed;
}

// F1 (unless a producer already wrote packed_x), F2 (unless the layer's cache holds Q(W)), F3: y [T, O]
Tensor forward_products(const Layer& l, const Tensor& x2, const Tensor& weight, at::ScalarType out_dtype, Tensor& packed_x, Tensor& packed_w) {
    const Tensor w2 = weight.contiguous();
    int flags = (packed_x.defined() ? QM_X_IS_PACKED : 0) | (packed_w.defined() ? QM_W_IS_PACKED : 0);
    Tensor xq_in = x2;
    if (l.x_dense.defined() && !packed_x.defined()) {
        packed_x = quantize_dense_into_packed(x2, l.x_dense, l.layout);
        flags |= QM_X_IS_PACKED;
    }
    if (l.w_dense.defined() && !packed_w.defined()) {
        packed_w = quantize_dense_into_packed(w2, l.w_dense, l.layout);
        flags |= QM_W_IS_PACKED;
    }
    if (flags & QM_X_IS_PACKED) xq_in = Tensor();
    if (!packed_x.defined()) packed_x = packed_buffer(l.T, l.I, w2);
    if (!packed_w.defined()) packed_w = packed_buffer(l.O, l.I, w2);
    Tensor y = at::empty({l.T, l.O}, w2.options().dtype(out_dtype));
    check(qm_linear_forward(ptr(xq_in), xq_in.defined() ? dtype_code(xq_in.scalar_type()) : 0, w2.data_ptr(), dtype_code(w2.scalar_type()),
                            l.T, l.I, l.O, l.a_hd, l.a_signs.data(), l.w_hd, l.w_signs.data(), packed_x.data_ptr(), (size_t)packed_x.numel(),
                            packed_w.data_ptr(), (size_t)packed_w.numel(), flags, y.data_ptr(), dtype_code(out_dtype), l.layout,
                            stream_of(w2)),
          "qm_linear_forward");
    return y;
}

// Whether a producer's grid quantizes the layer's weight along: it is not packed yet, fp32, aligned, under a Hadamard block of 32
bool takes_weight(const Layer& l, const Tensor& weight, const Tensor* packed_w) {
    return packed_w && !packed_w->defined() && l.T > 0 && l.layout == QM_LAYOUT_PADDED && l.w_hd == 32 && !l.w_dense.defined() && weight.scalar_type() == at::kFloat &&
           weight.is_contiguous() && reinterpret_cast<uintptr_t>(weight.data_ptr()) % 16 == 0;
}

// Straight-through backward of a forward quantizer with a dense rotation: (g * clip mask) @ matrix^T per group of 32, in
// g's dtype like the module path's product.
Tensor dense_rotation_backward(const Tensor& g, const Tensor& maskbits, const Tensor& dense, at::ScalarType x_dtype, at::ScalarType scale_dtype) {
    const Tensor shifts = at::arange(8, maskbits.options());
    const Tensor keep = maskbits.unsqueeze(-1).bitwise_right_shift(shifts).bitwise_and(1).view(g.sizes()).to(g.scalar_type());
    const Tensor m = dense.to(g.device()).to(x_dtype).to(at::kFloat).to(scale_dtype).to(g.scalar_type());
    return at::matmul((g * keep).reshape({-1, 32}), m.t()).view(g.sizes());
}

struct Gradients {
    Tensor gx, gw;
    at::ScalarType x_scale;   // dtype whose rounding of 32^-1/2 the activation quantizer's matrix carries in backward
};

// B1-B8: e [.., O] -> gradients w.r.t. the tensor F1 quantized [T, I] and w.r.t. W [O, I].  With gx_rotated, B7 is left to
// the kernel that consumes gx.
Gradients backward_products(const Layer& l, const Tensor& e, const Tensor& packed_x, const Tensor& packed_w, bool gx_rotated) {
    const bool low = autocast_bf16() || e.scalar_type() == at::kBFloat16;
    const at::ScalarType mid = low ? at::kBFloat16 : e.scalar_type();
    const at::ScalarType sd_x = low ? at::kBFloat16 : l.x_dtype, sd_w = low ? at::kBFloat16 : l.w_dtype;
    const Tensor e2 = rows_of(e, e.size(-1));
    require_cuda(e2);
    Signs g_signs;
    uint64_t seeds[4];
    bool stochastic;
    Tensor matrix, seed_base;
    {
        py::gil_scoped_acquire gil;
        try {
            const py::tuple drawn = py::reinterpret_steal<py::object>(PyObject_CallFunction(
                g_draw, "OOLLL", l.g_q.p, l.seed_base_ok ? Py_True : Py_False, (long long)l.T, (long long)l.I, (long long)l.O));
            if (!drawn.ptr()) throw py::error_already_set();
            g_signs = signs_of(drawn[0]);
            const py::tuple s = drawn[1];
            for (int i = 0; i < 4; ++i) seeds[i] = s[i].cast<uint64_t>();
            stochastic = drawn[2].cast<bool>();
            if (!drawn[3].is_none()) matrix = drawn[3].cast<Tensor>().to(e2.device(), at::kFloat).contiguous();
            if (!drawn[4].is_none()) seed_base = drawn[4].cast<Tensor>();
        } catch (py::error_already_set& err) {
            err.restore();
            python_error again;
            again.persist();
            throw again;
        }
    }
    const bool w_rotated = l.w_dense.defined(), x_rotated = gx_rotated || l.x_dense.defined();
    const int mid_code = dtype_code(mid);
    const at::ScalarType gw_dtype = mid == at::kBFloat16 && !w_rotated && (l.w_dtype == at::kFloat || l.w_dtype == at::kBFloat16) ? l.w_dtype : mid;
    const int64_t nbytes = (int64_t)qm_linear_backward_workspace_bytes(l.T, l.I, l.O, mid_code);
    const Tensor work = bytes(nbytes, e2);
    Tensor gx = at::empty({l.T, l.I}, e2.options().dtype(mid)), gw = at::empty({l.O, l.I}, e2.options().dtype(gw_dtype));
    check(qm_linear_backward_seeded(e2.data_ptr(), dtype_code(e2.scalar_type()), l.T, l.I, l.O, packed_x.data_ptr(), packed_w.data_ptr(),
                                    l.a_hd, l.a_signs.data(), l.w_hd, l.w_signs.data(), l.g_hd, g_signs.data(),
                                    stochastic ? QM_ABSMAX_SR : QM_ABSMAX_RTN, seeds, dtype_code(l.x_dtype), dtype_code(l.w_dtype), mid_code,
                                    dtype_code(sd_x), dtype_code(sd_w), work.data_ptr(), (size_t)nbytes, gx.data_ptr(), gw.data_ptr(),
                                    dtype_code(gw_dtype), l.layout, (x_rotated ? QM_GX_ROTATED : 0) | (w_rotated ? QM_GW_ROTATED : 0),
                                    matrix.defined() ? matrix.data_ptr<float>() : nullptr,
                                    seed_base.defined() ? reinterpret_cast<const uint64_t*>(seed_base.data_ptr<int64_t>()) : nullptr, stream_of(e2)),
          "qm_linear_backward");
    if (w_rotated) gw = dense_rotation_backward(gw, mask_bits(packed_w, l.O, l.I), l.w_dense, l.w_dtype, sd_w);
    if (l.x_dense.defined() && !gx_rotated) gx = dense_rotation_backward(gx, mask_bits(packed_x, l.T, l.I), l.x_dense, l.x_dtype, sd_x);
    return {gx, gw, sd_x};
}

// The same for the error-only scheme (backward.py:21-45): Q(e) and Q(e^T) times the packed operands as they are, in bf16
Gradients error_products(const Layer& l, const Tensor& e, const Tensor& packed_x, const Tensor& packed_w) {
    const Tensor e2 = rows_of(e, e.size(-1));
    require_cuda(e2);
    Signs g_signs;
    uint64_t seeds[2];
    bool stochastic;
    {
        py::gil_scoped_acquire gil;
        try {
            const py::tuple drawn = py::reinterpret_steal<py::object>(PyObject_CallFunctionObjArgs(g_error_draw, l.g_q.p, py::cast(e2).ptr(), nullptr));
            if (!drawn.ptr()) throw py::error_already_set();
            g_signs = signs_of(drawn[0]);
            const py::tuple s = drawn[1];
            for (int i = 0; i < 2; ++i) seeds[i] = s[i].cast<uint64_t>();
            stochastic = drawn[2].cast<bool>();
        } catch (py::error_already_set& err) {
            err.restore();
            python_error again;
            again.persist();
            throw again;
        }
    }
    const at::ScalarType gw_dtype = l.w_dtype == at::kFloat ? at::kFloat : at::kBFloat16;
    const int64_t nbytes = (int64_t)qm_linear_backward_error_workspace_bytes(l.T, l.I, l.O);
    const Tensor work = bytes(nbytes, e2);
    const Tensor gx = at::empty({l.T, l.I}, e2.options().dtype(at::kBFloat16)), gw = at::empty({l.O, l.I}, e2.options().dtype(gw_dtype));
    check(qm_linear_backward_error(e2.data_ptr(), dtype_code(e2.scalar_type()), l.T, l.I, l.O, packed_x.data_ptr(), packed_w.data_ptr(), l.a_hd,
                                   l.a_signs.data(), l.w_hd, l.w_signs.data(), l.g_hd, g_signs.data(), stochastic ? QM_ABSMAX_SR : QM_ABSMAX_RTN,
                                   seeds, QM_BF16, QM_BF16, work.data_ptr(), (size_t)nbytes, gx.data_ptr(), gw.data_ptr(), dtype_code(gw_dtype),
                                   stream_of(e2)),
          "qm_linear_backward_error");
    return {gx, gw, at::kBFloat16};
}

void keep_layer(AutogradContext* ctx, const LayerPtr& l) { ctx->saved_data["layer"] = c10::IValue::make_capsule(l); }
LayerPtr kept_layer(AutogradContext* ctx) { return c10::static_intrusive_pointer_cast<Layer>(ctx->saved_data["layer"].toCapsule()); }

// ---- y = Q(x) Q(W)^T with the fully quantized backward (backward.py:57-85, quantizers/mxfp4.py:143-146) ------------
Tensor linear_forward(const LayerPtr& l, const Tensor& x, const Tensor& weight, Tensor& packed_x, Tensor& packed_w) {
    require_cuda(x, weight);
    const Tensor x2 = rows_of(x, weight.size(1));
    set_extents(*l, x2.size(0), weight);
    l->x_dtype = x.scalar_type();
    const Tensor y = forward_products(*l, x2, weight, autocast_bf16() ? at::kBFloat16 : x.scalar_type(), packed_x, packed_w);
    auto shape = x.sizes().vec();
    shape.back() = l->O;
    return y.view(shape);
}
// A decoded batch against a weight that is already packed: one launch, undefined where that kernel does not serve
Tensor linear_decode(const Layer& l, const Tensor& x, const Tensor& weight, const Tensor& packed_w) {
    const int64_t I = weight.size(1), O = weight.size(0);
    if (x.numel() == 0 || x.numel() > 16 * I || l.a_hd != 32 || l.x_dense.defined() || l.w_dense.defined() || x.size(-1) != I || O >= kLongContraction) return {};
    const int64_t T = x.numel() / I;
    if (!qm_linear_decode_serves(T, I, O)) return {};
    require_cuda(x, weight);
    const Tensor x2 = rows_of(x, I);
    if (reinterpret_cast<uintptr_t>(x2.data_ptr()) % 16) return {};
    auto shape = x.sizes().vec();
    shape.back() = O;
    const at::ScalarType out_dtype = autocast_bf16() ? at::kBFloat16 : x.scalar_type();
    Tensor y = at::empty(shape, weight.options().dtype(out_dtype));
    check(qm_linear_decode(x2.data_ptr(), dtype_code(x2.scalar_type()), T, I, O, l.a_signs.data(), packed_w.data_ptr(), (size_t)packed_w.numel(),
                           y.data_ptr(), dtype_code(out_dtype), stream_of(x2)),
          "qm_linear_decode");
    return y;
}
struct LinearFn : Function<LinearFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const LayerPtr& l, Tensor* packed_w) {
        Tensor packed_x;
        const Tensor y = linear_forward(l, x, weight, packed_x, *packed_w);
        ctx->save_for_backward({packed_x, *packed_w});
        l->x_shape = x.sizes().vec();
        keep_layer(ctx, l);
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const LayerPtr l = kept_layer(ctx);
        const auto saved = ctx->get_saved_variables();
        const c10::OptionalDeviceGuard guard(saved[0].device());
        const Gradients g = l->error_only ? error_products(*l, grads[0], saved[0], saved[1]) : backward_products(*l, grads[0], saved[0], saved[1], false);
        return {g.gx.to(l->x_dtype).view(l->x_shape), g.gw.to(l->w_dtype), Tensor(), Tensor()};
    }
};
bool wants_grad(std::initializer_list<const Tensor*> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}

py::tuple linear(const Tensor& x, const Tensor& weight, int a_hd, py::handle a_signs, int w_hd, py::handle w_signs, int g_hd, py::handle g_q,
                 const optional<Tensor>& packed_weight, const optional<Tensor>& x_dense, const optional<Tensor>& w_dense, bool error_only) {
    return from_python([&] {
        const LayerPtr l = make_layer(a_hd, a_signs, w_hd, w_signs, g_hd, g_q, x_dense, w_dense);
        l->error_only = error_only;
        Tensor packed_w = or_none(packed_weight), packed_x;
        const c10::OptionalDeviceGuard guard(weight.is_cuda() ? std::optional<at::Device>(weight.device()) : std::nullopt);
        Tensor y;
        if (wants_grad({&x, &weight})) y = LinearFn::apply(x, weight, l, &packed_w);
        else if (packed_w.defined()) y = linear_decode(*l, x, weight, packed_w);
        if (!y.defined()) y = linear_forward(l, x, weight, packed_x, packed_w);
        return py::make_tuple(y, packed_w);
    });
}

// ---- the layer behind an RMSNorm --------------------------------------------------------------------------------------
// y = Q(rmsnorm(x) * gain) Q(W)^T; backward = the layer's quantized backward followed by RMSNorm's, which takes B7 with it.
// The second output is x itself (pass_input) or x + add, formed inside the quantizer kernel: the caller's residual sum
// continues with it, so both gradients of x arrive here together.
struct NormArgs {
    double eps;
    bool has_add, pass_input;
    Tensor* packed_w;
};
// Q(rmsnorm(x2 [+ add2]) * gain) as the layer's packed operand; x2 becomes the sum
// packed_w: where the layer's weight goes along, undefined on entry (see takes_weight)
Tensor normed_into_packed(const Layer& l, Tensor& x2, const Tensor& add2, const Tensor& gain, double eps, Tensor& factor, const Tensor& weight = Tensor(),
                          Tensor* packed_w = nullptr) {
    Tensor packed_x = packed_buffer(l.T, l.I, x2), x_sum;
    factor = at::empty({l.T}, x2.options().dtype(at::kFloat));
    if (add2.defined()) x_sum = at::empty_like(x2);
    if (takes_weight(l, weight, packed_w) && x2.scalar_type() == at::kFloat && (!add2.defined() || add2.scalar_type() == at::kBFloat16)) {
        *packed_w = packed_buffer(l.O, l.I, weight);
        check(qm_rmsnorm_quantize_with_weight_mxfp4(x2.data_ptr(), QM_F32, ptr(add2), QM_BF16, add2.defined() ? x_sum.data_ptr() : nullptr, gain.data_ptr<float>(),
                                                    (float)eps, l.T, l.I, l.a_signs.data(), packed_x.data_ptr(), (size_t)packed_x.numel(), factor.data_ptr<float>(),
                                                    weight.data_ptr<float>(), l.O, l.w_signs.data(), packed_w->data_ptr(), (size_t)packed_w->numel(), stream_of(x2)),
              "qm_rmsnorm_quantize_with_weight_mxfp4");
    } else {
        check(qm_rmsnorm_quantize_mxfp4(x2.data_ptr(), dtype_code(x2.scalar_type()), ptr(add2), add2.defined() ? dtype_code(add2.scalar_type()) : 0,
                                        add2.defined() ? x_sum.data_ptr() : nullptr, gain.data_ptr<float>(), (float)eps, l.T, l.I, l.a_signs.data(),
                                        packed_x.data_ptr(), (size_t)packed_x.numel(), factor.data_ptr<float>(), l.layout, stream_of(x2)),
              "qm_rmsnorm_quantize_mxfp4");
    }
    if (add2.defined()) x2 = x_sum;
    return packed_x;
}
struct NormLinearFn : Function<NormLinearFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const optional<Tensor>& add_in, const Tensor& gain,
                                 const Tensor& weight, const LayerPtr& l, const NormArgs& args) {
        const Tensor add = or_none(add_in);
        require_cuda(x, gain, weight, add);
        const int64_t I = weight.size(1);
        Tensor x2 = rows_of(x, I);
        set_extents(*l, x2.size(0), weight);
        l->x_dtype = at::kFloat;   // the normalised tensor times the fp32 gain is an fp32 tensor
        const Tensor gain_c = gain.contiguous();
        Tensor factor;
        Tensor packed_x = normed_into_packed(*l, x2, args.has_add ? rows_of(add, I) : Tensor(), gain_c, args.eps, factor, weight, args.packed_w);
        Tensor y = forward_products(*l, Tensor(), weight, autocast_bf16() ? at::kBFloat16 : at::kFloat, packed_x, *args.packed_w);
        if (ctx) {
            ctx->set_materialize_grads(false);
            ctx->save_for_backward({x2, gain_c, factor, packed_x, *args.packed_w});
            l->x_shape = x.sizes().vec();
            keep_layer(ctx, l);
            ctx->saved_data["add"] = args.has_add ? (int64_t)add.scalar_type() : (int64_t)-1;
        }
        auto shape = x.sizes().vec();
        shape.back() = l->O;
        y = y.view(shape);
        if (args.has_add) return {y, x2.view(x.sizes())};
        if (args.pass_input) return {y, x};
        return {y};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const LayerPtr l = kept_layer(ctx);
        const auto saved = ctx->get_saved_variables();
        const Tensor &x2 = saved[0], &gain = saved[1], &factor = saved[2], &packed_x = saved[3], &packed_w = saved[4];
        const c10::OptionalDeviceGuard guard(x2.device());
        Tensor e = grads[0];
        if (!e.defined()) e = at::zeros({l->T, l->O}, x2.options().dtype(at::kBFloat16));
        const Gradients g = backward_products(*l, e, packed_x, packed_w, true);
        Tensor skip;
        if (grads.size() > 1 && grads[1].defined()) skip = grads[1].reshape(x2.sizes()).to(x2.scalar_type()).contiguous();
        const int64_t add_type = ctx->saved_data["add"].toInt();
        const bool bf16_copy = add_type == (int64_t)at::kBFloat16;
        const Tensor mask = mask_bits(packed_x, l->T, l->I);
        const size_t nbytes = qm_rmsnorm_backward_workspace_bytes(l->T, l->I);
        const Tensor work = bytes(std::max<int64_t>((int64_t)nbytes, 1), x2);
        Tensor dx = at::empty_like(x2), dgain = at::empty({l->I}, x2.options().dtype(at::kFloat)), dx_bf16;
        if (bf16_copy) dx_bf16 = at::empty(x2.sizes(), x2.options().dtype(at::kBFloat16));
        check(qm_rmsnorm_backward(g.gx.data_ptr(), dtype_code(g.gx.scalar_type()), x2.data_ptr(), dtype_code(x2.scalar_type()),
                                  gain.data_ptr<float>(), factor.data_ptr<float>(), l->T, l->I, mask.data_ptr<uint8_t>(), l->a_signs.data(),
                                  dtype_code(g.x_scale), ptr(skip), dx.data_ptr(), bf16_copy ? dx_bf16.data_ptr() : nullptr, dgain.data_ptr<float>(),
                                  work.data_ptr(), nbytes, stream_of(x2)),
              "qm_rmsnorm_backward");
        dx = dx.view(l->x_shape);
        const Tensor d_add = add_type < 0 ? Tensor() : bf16_copy ? dx_bf16.view(l->x_shape) : dx;
        return {dx, d_add, dgain, g.gw.to(l->w_dtype), Tensor(), Tensor()};
    }
};
py::tuple norm_linear(const Tensor& x, const optional<Tensor>& add, const Tensor& gain, const Tensor& weight, double eps, py::handle a_signs,
                      int w_hd, py::handle w_signs, int g_hd, py::handle g_q, const optional<Tensor>& packed_weight,
                      const optional<Tensor>& w_dense, bool pass_input) {
    return from_python([&] {
        const LayerPtr l = make_layer(32, a_signs, w_hd, w_signs, g_hd, g_q, std::nullopt, w_dense);
        Tensor packed_w = or_none(packed_weight);
        const Tensor add_t = or_none(add);
        const NormArgs args{eps, add_t.defined(), pass_input, &packed_w};
        const c10::OptionalDeviceGuard guard(weight.device());
        const variable_list out = wants_grad({&x, &add_t, &gain, &weight}) ? NormLinearFn::apply(x, add, gain, weight, l, args)
                                                                           : NormLinearFn::forward(nullptr, x, add, gain, weight, l, args);
        return py::make_tuple(out[0], out.size() > 1 ? py::cast(out[1]) : py::none(), packed_w);
    });
}

// ---- the layer behind a SwiGLU: y = Q(silu(up) * gate) Q(W)^T with h12 = (up, gate) ----------------------------------
struct SwigluLinearFn : Function<SwigluLinearFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& h12, const Tensor& weight, const LayerPtr& l, Tensor* packed_w) {
        require_cuda(h12, weight);
        const int64_t I = weight.size(1);
        const Tensor h2 = rows_of(h12, 2 * I);
        set_extents(*l, h2.size(0), weight);
        l->x_dtype = h12.scalar_type();
        Tensor packed_x = packed_buffer(l->T, I, h2);
        if (takes_weight(*l, weight, packed_w) && h2.scalar_type() == at::kBFloat16) {
            *packed_w = packed_buffer(l->O, I, weight);
            check(qm_swiglu_quantize_with_weight_mxfp4(h2.data_ptr(), QM_BF16, l->T, I, l->a_signs.data(), packed_x.data_ptr(), (size_t)packed_x.numel(),
                                                       weight.data_ptr<float>(), l->O, l->w_signs.data(), packed_w->data_ptr(), (size_t)packed_w->numel(),
                                                       stream_of(h2)),
                  "qm_swiglu_quantize_with_weight_mxfp4");
        } else {
            check(qm_swiglu_quantize_mxfp4(h2.data_ptr(), dtype_code(h2.scalar_type()), l->T, I, l->a_signs.data(), packed_x.data_ptr(),
                                           (size_t)packed_x.numel(), l->layout, stream_of(h2)),
                  "qm_swiglu_quantize_mxfp4");
        }
        const Tensor y = forward_products(*l, Tensor(), weight, autocast_bf16() ? at::kBFloat16 : h12.scalar_type(), packed_x, *packed_w);
        if (ctx) {
            ctx->save_for_backward({h2, packed_x, *packed_w});
            l->x_shape = h12.sizes().vec();
            keep_layer(ctx, l);
        }
        auto shape = h12.sizes().vec();
        shape.back() = l->O;
        return y.view(shape);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const LayerPtr l = kept_layer(ctx);
        const auto saved = ctx->get_saved_variables();
        const Tensor &h2 = saved[0], &packed_x = saved[1], &packed_w = saved[2];
        const c10::OptionalDeviceGuard guard(h2.device());
        const Gradients g = backward_products(*l, grads[0], packed_x, packed_w, true);
        const Tensor mask = mask_bits(packed_x, l->T, l->I);
        Tensor d = at::empty_like(h2);
        check(qm_swiglu_backward(g.gx.data_ptr(), dtype_code(g.gx.scalar_type()), h2.data_ptr(), dtype_code(h2.scalar_type()), l->T, l->I,
                                 mask.data_ptr<uint8_t>(), l->a_signs.data(), dtype_code(g.x_scale), d.data_ptr(), stream_of(h2)),
              "qm_swiglu_backward");
        return {d.view(l->x_shape), g.gw.to(l->w_dtype), Tensor(), Tensor()};
    }
};
py::tuple swiglu_linear(const Tensor& h12, const Tensor& weight, py::handle a_signs, int w_hd, py::handle w_signs, int g_hd, py::handle g_q,
                        const optional<Tensor>& packed_weight, const optional<Tensor>& w_dense) {
    return from_python([&] {
        const LayerPtr l = make_layer(32, a_signs, w_hd, w_signs, g_hd, g_q, std::nullopt, w_dense);
        Tensor packed_w = or_none(packed_weight);
        const c10::OptionalDeviceGuard guard(weight.device());
        const Tensor y = wants_grad({&h12, &weight}) ? SwigluLinearFn::apply(h12, weight, l, &packed_w)
                                                     : SwigluLinearFn::forward(nullptr, h12, weight, l, &packed_w);
        return py::make_tuple(y, packed_w);
    });
}

// ---- rotary split of the fused attention projection (llama.py:43-61) and its merge in backward -----------------------
struct RopeFn : Function<RopeFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& table, int64_t n_head) {
        const int64_t B = qkv.size(0), S = qkv.size(1), C = qkv.size(2) / 3, hs = C / n_head;
        // the reference rotates in fp32 and autocast hands attention bf16 copies: one rounding of the fp32 result
        const at::ScalarType out_dtype = autocast_bf16() ? at::kBFloat16 : at::kFloat;
        const Tensor in = rows_of(qkv, 3 * C);
        Tensor out[3];
        for (Tensor& t : out) t = at::empty({B, S, n_head, hs}, in.options().dtype(out_dtype));
        check(qm_rope_split_qkv(in.data_ptr(), dtype_code(in.scalar_type()), B * S, S, C, (int)hs, table.data_ptr<float>(), out[0].data_ptr(),
                                out[1].data_ptr(), out[2].data_ptr(), dtype_code(out_dtype), stream_of(in)),
              "qm_rope_split_qkv");
        if (ctx) {
            ctx->set_materialize_grads(false);
            ctx->save_for_backward({table});
            ctx->saved_data["shape"] = std::vector<int64_t>{B, S, C, hs, (int64_t)qkv.scalar_type()};
        }
        return {out[0], out[1], out[2]};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const Tensor table = ctx->get_saved_variables()[0];
        const auto s = ctx->saved_data["shape"].toIntVector();
        const int64_t B = s[0], S = s[1], C = s[2], hs = s[3];
        const at::ScalarType in_dtype = (at::ScalarType)s[4];
        const c10::OptionalDeviceGuard guard(table.device());
        at::ScalarType dt = at::kFloat;
        for (const Tensor& g : grads)
            if (g.defined()) { dt = g.scalar_type(); break; }
        Tensor flat[3];
        for (int i = 0; i < 3; ++i)
            flat[i] = grads[i].defined() ? grads[i].to(dt).contiguous() : at::zeros({B * S, C}, table.options().dtype(dt));
        Tensor d = at::empty({B, S, 3 * C}, table.options().dtype(in_dtype));
        check(qm_rope_merge_qkv_grad(flat[0].data_ptr(), flat[1].data_ptr(), flat[2].data_ptr(), dtype_code(dt), B * S, S, C, (int)hs,
                                     table.data_ptr<float>(), d.data_ptr(), dtype_code(in_dtype), stream_of(table)),
              "qm_rope_merge_qkv_grad");
        return {d, Tensor(), Tensor()};
    }
};
py::tuple rope_qkv(const Tensor& qkv, const Tensor& table, int64_t n_head) {
    return from_python([&] {
        require_cuda(qkv, table);
        const int64_t C = qkv.size(2) / 3;
        if (table.dim() != 3 || table.size(0) != qkv.size(1) || table.size(1) != C / n_head / 2 || table.size(2) != 2 || !table.is_contiguous())
            raise(PyExc_ValueError, "rope_qkv: table must be a contiguous [seq_len, head_dim / 2, 2] tensor");
        const c10::OptionalDeviceGuard guard(qkv.device());
        const variable_list out = wants_grad({&qkv}) ? RopeFn::apply(qkv, table, n_head) : RopeFn::forward(nullptr, qkv, table, n_head);
        return py::make_tuple(out[0], out[1], out[2]);
    });
}

// ---- evaluated models: layers behind an RMSNorm whose bf16 result feeds one kernel, which runs in the product's epilogue ------------
// Nothing is kept for a backward pass.  Packed weights are given; where a kernel does not serve, None comes back and nothing was launched.
py::object norm_swiglu_linear(const Tensor& x, const optional<Tensor>& add, const Tensor& gain, double eps, const Tensor& w12, const Tensor& packed_w12,
                              py::handle a_signs12, const Tensor& w, const Tensor& packed_w, py::handle a_signs, int w_hd, py::handle w_signs) {
    return from_python([&]() -> py::object {
        const int64_t I = w12.size(1), hidden = w.size(1);
        const LayerPtr l = make_layer(32, a_signs12, 32, py::none(), 32, py::none(), std::nullopt, std::nullopt);
        const LayerPtr next = make_layer(32, a_signs, w_hd, w_signs, 32, py::none(), std::nullopt, std::nullopt);
        const Tensor add_t = or_none(add);
        require_cuda(x, gain, w12, w, add_t);
        const c10::OptionalDeviceGuard guard(w12.device());
        const int64_t T = x.numel() / I;
        if (x.size(-1) != I || gain.numel() != I || !qm_linear_swiglu_serves(T, I, hidden)) return py::none();
        set_extents(*l, T, w12);
        set_extents(*next, T, w);
        if (l->layout != QM_LAYOUT_PADDED || next->layout != QM_LAYOUT_PADDED || l->O != 2 * hidden) return py::none();
        Tensor x2 = rows_of(x, I), factor;
        Tensor packed_x = normed_into_packed(*l, x2, add_t.defined() ? rows_of(add_t, I) : Tensor(), gain.contiguous(), eps, factor);
        Tensor packed_h = packed_buffer(T, hidden, x2), packed = packed_w;
        check(qm_linear_swiglu_quantize(packed_x.data_ptr(), (size_t)packed_x.numel(), packed_w12.data_ptr(), (size_t)packed_w12.numel(), T, I, hidden,
                                        next->a_signs.data(), packed_h.data_ptr(), (size_t)packed_h.numel(), stream_of(x2)),
              "qm_linear_swiglu_quantize");
        const Tensor y = forward_products(*next, Tensor(), w, at::kBFloat16, packed_h, packed);
        auto shape = x.sizes().vec();
        shape.back() = next->O;
        return py::make_tuple(y.view(shape), add_t.defined() ? x2.view(x.sizes()) : x);
    });
}
py::object norm_rope_linear(const Tensor& x, const optional<Tensor>& add, const Tensor& gain, double eps, const Tensor& weight, const Tensor& packed_w,
                            py::handle a_signs, const Tensor& table, int64_t n_head) {
    return from_python([&]() -> py::object {
        const int64_t I = weight.size(1), C = weight.size(0) / 3, hs = C / n_head;
        const LayerPtr l = make_layer(32, a_signs, 32, py::none(), 32, py::none(), std::nullopt, std::nullopt);
        const Tensor add_t = or_none(add);
        require_cuda(x, gain, weight, table, add_t);
        const c10::OptionalDeviceGuard guard(weight.device());
        const int64_t T = x.numel() / I;
        if (x.dim() != 3 || x.size(2) != I || gain.numel() != I || weight.size(0) != 3 * C || !qm_linear_rope_serves(T, I, C, (int)hs)) return py::none();
        const int64_t B = x.size(0), S = x.size(1);
        if (table.dim() != 3 || table.size(0) != S || table.size(1) != hs / 2 || table.size(2) != 2 || !table.is_contiguous() ||
            reinterpret_cast<uintptr_t>(table.data_ptr()) % 16)
            return py::none();
        set_extents(*l, T, weight);
        if (l->layout != QM_LAYOUT_PADDED) return py::none();
        Tensor x2 = rows_of(x, I), factor;
        Tensor packed_x = normed_into_packed(*l, x2, add_t.defined() ? rows_of(add_t, I) : Tensor(), gain.contiguous(), eps, factor);
        Tensor out[3];
        for (Tensor& t : out) t = at::empty({B, S, n_head, hs}, x2.options().dtype(at::kBFloat16));
        check(qm_linear_rope(packed_x.data_ptr(), (size_t)packed_x.numel(), packed_w.data_ptr(), (size_t)packed_w.numel(), T, I, C, (int)hs, S,
                             table.data_ptr<float>(), out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), stream_of(x2)),
              "qm_linear_rope");
        return py::make_tuple(out[0], out[1], out[2], add_t.defined() ? x2.view(x.sizes()) : x);
    });
}

// ---- quantizer modules: pseudo-quantized tensor forward, straight-through backward (quantizers/mxfp4.py:15-34,127-146)
struct QuantizerArgs {
    int hd, mode;
    Signs signs;
    uint64_t seed;
    double post;
};
// contiguous 2-D view whose rows are whole Hadamard chunks
Tensor chunk_rows(const Tensor& x, int64_t hd) {
    const Tensor c = x.contiguous();
    const int64_t last = c.dim() > 0 ? c.size(-1) : 1;
    return c.view({-1, c.dim() > 0 && last % hd == 0 ? last : hd});   // raises if the element count is not a multiple of hd
}
struct QuantizerFn : Function<QuantizerFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const QuantizerArgs& a) {
        require_cuda(x);
        const Tensor x2 = chunk_rows(x, a.hd);
        const int64_t rows = x2.size(0), cols = x2.size(1);
        const bool quest = a.mode == QM_QUEST_RTN || a.mode == QM_QUEST_SR;
        Tensor mask, deq = at::empty({rows, cols}, x2.options());
        if (quest) mask = bytes(rows * cols / 8, x2);
        check(qm_pseudo_quantize_mxfp4(x2.data_ptr(), dtype_code(x2.scalar_type()), rows, cols, a.hd, a.signs.data(), a.mode, a.seed,
                                       quest ? mask.data_ptr<uint8_t>() : nullptr, deq.data_ptr(), stream_of(x2)),
              "qm_pseudo_quantize_mxfp4");
        if (a.post != 1.0) deq.mul_(a.post);
        if (ctx) {
            if (quest) ctx->save_for_backward({mask});
            ctx->saved_data["shape"] = x.sizes().vec();
            ctx->saved_data["meta"] = std::vector<int64_t>{rows, cols, a.hd, (int64_t)x.scalar_type(), a.signs.w[0], a.signs.w[1], a.signs.w[2], a.signs.w[3], quest};
        }
        return deq.view(x.sizes());
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto m = ctx->saved_data["meta"].toIntVector();
        // asked for only where something was saved: a graph that keeps no tensor can be gone through again
        const Tensor mask = m[8] ? ctx->get_saved_variables()[0] : Tensor();
        const at::ScalarType x_dtype = (at::ScalarType)m[3];
        Signs signs;
        for (int i = 0; i < 4; ++i) signs.w[i] = (uint32_t)m[4 + i];
        const Tensor g = grads[0].contiguous().view({m[0], m[1]});
        const c10::OptionalDeviceGuard guard(g.device());
        // under bf16 autocast the reference's `g @ H.T` runs with H cast to bf16 and a bf16 result
        const bool low = autocast_bf16() || g.scalar_type() == at::kBFloat16;
        const at::ScalarType out_dtype = low ? at::kBFloat16 : g.scalar_type();
        Tensor out = at::empty({m[0], m[1]}, g.options().dtype(out_dtype));
        check(qm_masked_hadamard_bwd(g.data_ptr(), dtype_code(g.scalar_type()), m[0], m[1], (int)m[2], dtype_code(low ? at::kBFloat16 : x_dtype),
                                     signs.data(), m[8] ? mask.data_ptr<uint8_t>() : nullptr, out.data_ptr(), dtype_code(out_dtype),
                                     stream_of(g)),
              "qm_masked_hadamard_bwd");
        return {out.view(ctx->saved_data["shape"].toIntVector()).to(x_dtype), Tensor()};
    }
};
Tensor quantizer(const Tensor& x, int hd, py::handle signs, int mode, uint64_t seed, double post) {
    return from_python([&] {
        const QuantizerArgs a{hd, mode, signs_of(signs), seed, post};
        const c10::OptionalDeviceGuard guard(x.is_cuda() ? std::optional<at::Device>(x.device()) : std::nullopt);
        return wants_grad({&x}) ? QuantizerFn::apply(x, a) : QuantizerFn::forward(nullptr, x, a);
    });
}

// `hd` fresh sign flips of re_randomize("signs"): the draw of torch.randint(0, 2, (hd,)) from the default host generator
// (the same stream), as a bit mask with bit j set where the draw was 0, i.e. where column j flips
py::int_ sign_flips(int64_t hd) {
    const Tensor flips = at::randint(0, 2, {hd}, at::TensorOptions().dtype(at::kLong));
    const int64_t* f = flips.data_ptr<int64_t>();
    unsigned char raw[16] = {};
    for (int64_t j = 0; j < hd && j < 128; ++j)
        if (f[j] == 0) raw[j >> 3] |= (unsigned char)(1u << (j & 7));
    return py::reinterpret_steal<py::int_>(_PyLong_FromByteArray(raw, sizeof(raw), 1, 0));
}

// quartet_amd.one_node.transformed() in one call without arguments (0.03 us; every layer call asks)
PyObject* transformed(PyObject*, PyObject*) {
    const bool yes = torch::jit::tracer::isTracing() || torch::autograd::ForwardADLevel::try_get_by_idx(0) ||
                     c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
    return PyBool_FromLong(yes);
}
PyMethodDef transformed_def = {"transformed", transformed, METH_NOARGS, nullptr};

void bind(py::object error_class, py::object draw, py::object error_draw) {
    g_error_class = error_class.release().ptr();
    g_draw = draw.release().ptr();
    g_error_draw = error_draw.release().ptr();
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("bind", &bind);
    m.def("linear", &linear);
    m.def("norm_linear", &norm_linear);
    m.def("swiglu_linear", &swiglu_linear);
    m.def("rope_qkv", &rope_qkv);
    m.def("norm_swiglu_linear", &norm_swiglu_linear);
    m.def("norm_rope_linear", &norm_rope_linear);
    m.def("quantizer", &quantizer);
    m.def("sign_flips", &sign_flips);
    m.add_object("transformed", py::reinterpret_steal<py::object>(PyCFunction_New(&transformed_def, nullptr)));
}

// The Python operators' host path in native code: forward and backward of Linear, MLP and the variable-group linear for the
// standard recipes, as autograd nodes that marshal tensors into libviola_hip's entry points.
//
// Why it is native: a forward + backward of a small layer is a dozen kernels of 3-6 us each, and the Python marshalling
// around them (autograd.Function, one tensor per buffer, ctypes) took 130-200 us per step, three times the kernels. Here a
// pass allocates one arena per lifetime (scratch of the call, what is kept for backward) and carves raw pointers out of it,
// and backward runs on autograd's device thread without the interpreter.
//
// Row pitches: every GEMM operand made here has rows of a whole number of 128 k where its k axis is a token count (weight
// gradient), and of 16 k (128 under E8M0 scales) otherwise, padded with zero codes, and the GEMM takes the pitch as its k.
// Whatever the sizes, the kernels that load 16-byte pieces take the product. Their sums are the guarded kernel's but for the order
// in which the k range of a weight gradient is added: few tiles and a long k add two halves of it separately, or two to 64 parts
// (viola_group_gemm_parts). So with a token count that is no whole number of 16 one element in 10^4 of a weight gradient rounds the
// other way in 16 bits, and isolated momentum codes of an optimizer step behind it (1 in 10^5) and FP8 weights (0.2 to 0.5 %) take
// the neighbouring code.
#include "host.hpp"

#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

using namespace viola_host;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

namespace {

// ---------------------------------------------------------------------------------------------------- recipes
// State of one per-tensor quantizer, shared with its module and with nodes that advance it in backward: calls so far (its slot in
// the amax history), and whether its scale is that of the history (a checkpoint brings this along, so it may change). Atomic:
// backward counts on autograd's thread, without the interpreter's lock, while the program may read or set it.
struct Counter {
    std::atomic<int64_t> value;
    std::atomic<bool> delayed;
    Counter(int64_t value, bool delayed) : value(value), delayed(delayed) {}
};

// What a Linear's constructor fixed about its arithmetic. Standard recipes only: (1, 32) activation and gradient groups,
// (32, 32) weight blocks, FP32 accumulation, no rotation, FP8-saved inputs.
struct Recipe {
    bool grouped = false, native = false;      // native: E8M0 scales; not grouped: one FP32 scale per tensor
    bool fp8_weight = true, cache_transpose = false;
    int fwd = VIOLA_E4M3, bwd = VIOLA_E4M3;
    float fwd_limit = 448.0f, bwd_limit = 448.0f;
    int64_t in = 0, out = 0;

    explicit Recipe(const py::dict& d) {
        grouped = d["grouped"].cast<bool>(); native = d["native"].cast<bool>();
        fp8_weight = d["fp8_weight"].cast<bool>(); cache_transpose = d["cache_transpose"].cast<bool>();
        fwd = d["fwd"].cast<int>(); bwd = d["bwd"].cast<int>();
        fwd_limit = d["fwd_limit"].cast<float>(); bwd_limit = d["bwd_limit"].cast<float>();
        in = d["in"].cast<int64_t>(); out = d["out"].cast<int64_t>();
    }
    py::dict fields() const {                                    // for copies and pickles of a module
        using namespace py::literals;
        return py::dict("grouped"_a = grouped, "native"_a = native, "fp8_weight"_a = fp8_weight,
                        "cache_transpose"_a = cache_transpose, "fwd"_a = fwd, "bwd"_a = bwd, "fwd_limit"_a = fwd_limit, "bwd_limit"_a = bwd_limit,
                        "in"_a = in, "out"_a = out);
    }
    at::ScalarType codes() const { return fwd == VIOLA_E4M3 ? at::kFloat8_e4m3fn : at::kFloat8_e5m2; }
    at::ScalarType scales() const { return native ? at::kByte : at::kFloat; }
    int scale_format() const { return native ? VIOLA_SCALE_E8M0 : VIOLA_SCALE_F32; }
    int64_t scale_bytes() const { return native ? 1 : 4; }
    int64_t pitch(int64_t k) const { return native ? ceil_to(k, 128) : k % 16 == 0 ? k : ceil_to(k, 128); }
};

// The tensors of one Linear, fetched from the module for this call.
struct Layer {
    std::shared_ptr<Recipe> recipe;
    Tensor weight, bias, scale, transpose, transpose_scale;
    // per-tensor recipes: history and counter of the weight, input and gradient quantizers
    Tensor history[3];
    std::shared_ptr<Counter> counter[3];
};
enum { WEIGHT = 0, INPUT = 1, GRAD = 2 };

bool holds(const Tensor& t, const at::Device& device, at::ScalarType type, at::IntArrayRef sizes) {
    return t.defined() && t.device() == device && t.scalar_type() == type && t.sizes() == sizes && t.is_contiguous();
}

// Whether a framework transform is at work that sees operators and autograd functions, not these kernels: vmap, grad and the like
// (functorch), tracing, a dispatch mode written in Python.
bool transformed() {
    static const c10::DispatchKeySet keys({c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::Tracer, c10::DispatchKey::Python});
    return c10::impl::tls_local_dispatch_key_set().included_.has_any(keys);
}

// A tensor subclass with its own dispatch, or a dual number of forward-mode differentiation, whose tangent would be lost here.
bool plain(const Tensor& t) { return !t.defined() || (!t.unsafeGetTensorImpl()->is_python_dispatch() && !t._fw_grad(0).defined()); }

// Whether a layer's tensors are what the kernels here read by raw pointer: the recipe's formats and shapes, contiguous, on x's
// device, and plain. Any other call is the general path's (nn/_grouped_linear.py, nn/_tensor_linear.py), which copies a weight whose rows
// are not contiguous, follows the weight's own FP8 format and refuses what no kernel takes.
bool takes(const Layer& l, const at::Device& device) {
    const Recipe& r = *l.recipe;
    const int64_t rows = ceil_div(r.out, 32), cols = ceil_div(r.in, 32);
    const at::ScalarType stored = l.weight.scalar_type();
    if (r.fp8_weight ? stored != r.codes() : stored != at::kFloat && stored != at::kBFloat16 && stored != at::kHalf) return false;
    if (!plain(l.weight) || !plain(l.bias)) return false;
    if (r.in == 0 || r.out == 0 || !device.is_cuda() || !holds(l.weight, device, stored, {r.out, r.in})) return false;
    if (r.fp8_weight && !(r.grouped ? holds(l.scale, device, r.scales(), {rows, cols}) : holds(l.scale, device, at::kFloat, {1}))) return false;
    if (l.transpose.numel() && !(holds(l.transpose, device, r.codes(), {r.in, r.out}) && (!r.grouped || holds(l.transpose_scale, device, r.scales(), {cols, rows}))))
        return false;
    if (l.bias.defined() && (l.bias.device() != device || l.bias.numel() != r.out)) return false;
    if (!r.grouped)
        for (const Tensor& history : l.history)
            if (history.device() != device || history.scalar_type() != at::kFloat || !history.is_contiguous() || history.numel() == 0) return false;
    return true;
}

// Codes and scales of one operand; rows `pitch` codes apart.
struct Codes {
    const void* q = nullptr;
    const void* s = nullptr;
    int64_t pitch = 0;
};


// Where transposed codes and their scales lie in an arena; rows `pitch` codes apart.
struct Place {
    int64_t q = -1, s = -1, pitch = 0;
    Codes in(const void* base) const {
        const char* p = static_cast<const char*>(base);
        return q < 0 ? Codes{} : Codes{p + q, p + s, pitch};
    }
};

// A tensor that was saved for backward, as it comes back: a saved-tensor hook may have moved it or made another of it.
Tensor restored(const SavedVariable& saved, const at::Device& device, at::ScalarType type, at::IntArrayRef sizes) {
    const Tensor t = saved.unpack();
    TORCH_CHECK(t.defined() && t.device() == device && t.scalar_type() == type && t.sizes() == sizes, "a tensor saved by a viola module came back changed");
    return t.contiguous();
}

// What a projection's backward needs. All of it is saved the way autograd saves tensors, so that saved-tensor hooks (save_on_cpu,
// checkpointing) see it, in-place changes are noticed and it is freed with the graph; no address outlives the forward pass.
struct Kept {
    Arena arena;                                                 // forward only: transposed codes of the input, per-tensor scales
    Tensor weight_t, weight_t_scale;                             // forward only: the cached W^T, or this forward's
    Place input;                                                 // in the saved arena
    int64_t scales = -1;                                         // per-tensor recipes: the scale of x, then that of a 16-bit weight
    SavedVariable saved_arena, weight, weight_scale, saved_weight_t, saved_weight_t_scale;
    int64_t rows = 0;
    at::ScalarType x_dtype = at::kFloat, weight_grad = at::kFloat, bias_grad = at::kFloat;
    bool has_input = false, has_weight_t = false;

    // After the forward pass, where hooks run as they do for any operator: outside of its dispatch guard.
    void save(const Layer& l) {
        saved_arena = SavedVariable(arena.tensor(), false);
        weight = SavedVariable(l.weight, false);
        if (l.recipe->fp8_weight) weight_scale = SavedVariable(l.scale, false);
        has_weight_t = weight_t.defined() && weight_t.numel();
        if (has_weight_t) {
            saved_weight_t = SavedVariable(weight_t, false);
            if (l.recipe->grouped) saved_weight_t_scale = SavedVariable(weight_t_scale, false);
        }
        arena.release();
        weight_t = weight_t_scale = Tensor();
    }
    void release() {
        for (SavedVariable* v : {&saved_arena, &weight, &weight_scale, &saved_weight_t, &saved_weight_t_scale}) v->reset_data();
    }
};

// The tensors of one layer as its backward reads them.
struct Restored {
    Tensor arena, weight, weight_scale, weight_t, weight_t_scale;
    Codes input_t;
    const float* scales = nullptr;
};

Restored restore(const Kept& kept, const Recipe& r, const Tensor& dy) {
    const at::Device device = dy.device();
    const int64_t rows = ceil_div(r.out, 32), cols = ceil_div(r.in, 32);
    Restored t;
    t.weight = kept.weight.unpack();
    // the caller's tensor: it may have been moved or replaced (`.data`) since
    TORCH_CHECK(t.weight.device() == device && t.weight.sizes() == at::IntArrayRef({r.out, r.in}) && (!r.fp8_weight || t.weight.scalar_type() == r.codes()),
                "the weight of a viola Linear was moved or replaced between forward and backward");
    t.weight = t.weight.contiguous();
    if (kept.arena.size()) {
        t.arena = restored(kept.saved_arena, device, at::kByte, {kept.arena.size()});
        t.input_t = kept.input.in(t.arena.const_data_ptr());
        if (kept.scales >= 0) t.scales = reinterpret_cast<const float*>(static_cast<const char*>(t.arena.const_data_ptr()) + kept.scales);
    }
    if (r.fp8_weight) t.weight_scale = r.grouped ? restored(kept.weight_scale, device, r.scales(), {rows, cols}) : restored(kept.weight_scale, device, at::kFloat, {1});
    if (kept.has_weight_t) {
        t.weight_t = restored(kept.saved_weight_t, device, r.codes(), {r.in, r.out});
        if (r.grouped) t.weight_t_scale = restored(kept.saved_weight_t_scale, device, r.scales(), {cols, rows});
    }
    return t;
}

// ---------------------------------------------------------------------------------------------------- products
// Outputs the kernel for small products takes (viola_skinny_linear: one tile of 32 x 32 or less per CU, any width up to 32 rows), and
// up to which k (times two where a block has 32 rows) it quantizes x itself: every block does so again, which beyond costs more
// than the quantizer's launch (measured, 8 rows, 4096 wide: k = 1024 5.3 against 7.5 us, 4096 10.6 against 10.5, 8192 15.5 against
// 13.9). Per-tensor scales: every block reads the whole of x for its maximum.
constexpr int64_t QUANTIZED_IN_PRODUCT = 3072, WHOLE_TENSOR = 1 << 16;
bool small_product(int64_t m, int64_t n) { return m <= 32 || (m <= 4096 && ceil_div(m, 32) * ceil_div(n, 32) <= 256); }
// Codes between the rows of a product's operands: that kernel takes any whole number of 16-byte pieces.
int64_t product_pitch(const Recipe& r, int64_t m, int64_t n, int64_t k) { return k % 16 == 0 && small_product(m, n) ? k : r.pitch(k); }

// out[m, n] = a b^T, k = the operands' common pitch. br: rows of b per scale row (32: weight blocks, 1: row-wise).
void product(const Recipe& r, const Codes& a, int a_fmt, const Codes& b, int b_fmt, int64_t m, int64_t n, int br, const Tensor& bias,
             void* out, at::ScalarType out_dtype, const at::Device& device, viola_stream_t stream) {
    const int64_t k = a.pitch;
    TORCH_INTERNAL_ASSERT(b.pitch == k);
    const void* bias_p = ptr(bias);
    const int bias_code = bias_p ? code_of(bias.scalar_type()) : 0, out_code = code_of(out_dtype);
    if (br == 32 && small_product(m, n)) {
        const int status = VIOLA_TRY(viola_skinny_linear, a.q, a_fmt, static_cast<const float*>(a.s), m, k, b.q, b_fmt, b.s, r.grouped, n, r.fwd_limit,
                                     r.scale_format(), nullptr, 0, nullptr, bias_p, bias_code, out, out_code, stream);
        if (status == 0) return;
        if (status != VIOLA_EUNSUPPORTED) check("viola_skinny_linear", status);
    }
    if (!r.grouped) {
        VIOLA_CALL(viola_tensor_gemm, a.q, a_fmt, b.q, b_fmt, static_cast<const float*>(a.s), static_cast<const float*>(b.s), m, n, k, bias_p,
                   bias_code, out, out_code, stream);
        return;
    }
    const float *sa = static_cast<const float*>(a.s), *sb = static_cast<const float*>(b.s);
    Tensor decoded[2];
    if (r.native) {
        const int status = VIOLA_TRY(viola_mx_gemm, a.q, a_fmt, b.q, b_fmt, static_cast<const uint8_t*>(a.s), static_cast<const uint8_t*>(b.s), m, n,
                                     k, 1, br, bias_p, bias_code, out, out_code, stream);
        if (status == 0) return;
        if (status != VIOLA_EUNSUPPORTED) check("viola_mx_gemm", status);
        // operands beyond 2 GiB, which the block-scaled kernel declines: the same product with the scales spelled out in FP32
        const int64_t rows[2] = {m, ceil_div(n, br)};
        const void* bytes[2] = {a.s, b.s};
        for (int i = 0; i < 2; ++i) {
            const Tensor view = at::from_blob(const_cast<void*>(bytes[i]), {rows[i], ceil_div(k, 32)}, at::TensorOptions().dtype(at::kByte).device(device));
            decoded[i] = at::exp2(view.to(at::kFloat) - 127.0f);
        }
        sa = decoded[0].const_data_ptr<float>();
        sb = decoded[1].const_data_ptr<float>();
    }
    VIOLA_CALL(viola_group_gemm, a.q, a_fmt, b.q, b_fmt, sa, sb, m, n, k, 1, 32, br, 32, bias_p, bias_code, out, out_code, stream);
}

// The gated projections: forward aux = [g | u], out = act(g) * u (aux may be null); backward aux read, out = [d u act'(g) | d act(g)].
void gated_product(const Recipe& r, const Codes& a, int a_fmt, const Codes& b, int b_fmt, int64_t m, int64_t h, const Tensor& bias, const Tensor& aux_or_empty,
                   const Tensor& out, int activation, bool backward, viola_stream_t stream) {
    const int64_t k = a.pitch;
    TORCH_INTERNAL_ASSERT(b.pitch == k);
    const void* bias_p = ptr(bias);
    const int bias_code = bias_p ? code_of(bias.scalar_type()) : 0, dtype = code_of(out.scalar_type());
    void* aux = const_cast<void*>(ptr(aux_or_empty));
    void* to = const_cast<void*>(ptr(out));
    if (!r.grouped) {
        VIOLA_CALL(viola_tensor_gated_gemm, a.q, a_fmt, b.q, b_fmt, static_cast<const float*>(a.s), static_cast<const float*>(b.s), m, h, k, bias_p,
                   bias_code, aux, to, dtype, activation, backward, stream);
        return;
    }
    if (!r.native) {
        VIOLA_CALL(viola_gated_gemm, a.q, a_fmt, b.q, b_fmt, static_cast<const float*>(a.s), static_cast<const float*>(b.s), m, h, k, 1, 32, 32, 32,
                   bias_p, bias_code, aux, to, dtype, activation, backward, stream);
        return;
    }
    const int status = VIOLA_TRY(viola_mx_gated_gemm, a.q, a_fmt, b.q, b_fmt, static_cast<const uint8_t*>(a.s), static_cast<const uint8_t*>(b.s), m, h, k, 1,
                                 32, bias_p, bias_code, aux, to, dtype, activation, backward, stream);
    if (status == 0) return;
    if (status != VIOLA_EUNSUPPORTED) check("viola_mx_gated_gemm", status);
    // up rows off the scale grid (h not a multiple of 32): the same values from the plain product and the elementwise kernels
    if (backward) {
        const Tensor d = at::empty({m, h}, out.options());
        product(r, a, a_fmt, b, b_fmt, m, h, 32, Tensor(), d.mutable_data_ptr(), out.scalar_type(), out.device(), stream);
        VIOLA_CALL(viola_gated_backward, aux, ptr(d), to, m, h, dtype, activation, stream);
    } else {
        const Tensor z = aux ? aux_or_empty : at::empty({m, 2 * h}, out.options());
        product(r, a, a_fmt, b, b_fmt, m, 2 * h, 32, bias, z.mutable_data_ptr(), out.scalar_type(), out.device(), stream);
        VIOLA_CALL(viola_gated_forward, ptr(z), to, m, h, dtype, activation, stream);
    }
}

// ---------------------------------------------------------------------------------------------------- quantizers
// Row-wise and / or transposed codes of a grouped operand into reserved arena space.
struct GroupSpace {
    int64_t q = -1, s = -1, qt = -1, st = -1, pitch = 0, pitch_t = 0;
    void reserve(const Recipe& r, Arena* rowwise, Arena* transposed, int64_t rows, int64_t cols, int64_t row_pitch) {
        pitch = row_pitch;
        pitch_t = ceil_to(rows, 128);
        if (rowwise) { q = rowwise->take(rows * pitch); s = rowwise->take(rows * ceil_div(pitch, 32) * r.scale_bytes()); }
        if (transposed) { qt = transposed->take(cols * pitch_t); st = transposed->take(cols * (pitch_t / 32) * r.scale_bytes()); }
    }
};

void quantize_groups(const Recipe& r, const Tensor& x, int fmt, float limit, const GroupSpace& g, const Arena* rowwise, const Arena* transposed,
                     float* column_partial, Codes* out, Codes* out_t, viola_stream_t stream) {
    const int64_t rows = x.size(0), cols = x.size(1);
    void *q = nullptr, *s = nullptr, *qt = nullptr, *st = nullptr;
    if (g.q >= 0) { q = rowwise->at(g.q); s = rowwise->at(g.s); *out = {q, s, g.pitch}; }
    if (g.qt >= 0) { qt = transposed->at(g.qt); st = transposed->at(g.st); *out_t = {qt, st, g.pitch_t}; }
    const int dtype = code_of(x.scalar_type());
    if (!qt && g.pitch == cols)                                  // row-wise only: the streaming kernel
        VIOLA_CALL(viola_group_quantize, ptr(x), dtype, rows, cols, q, fmt, s, 1, 32, limit, 0, nullptr, 1, 32, r.scale_format(), stream);
    else
        VIOLA_CALL(viola_group_quantize_dual_pitched, ptr(x), dtype, rows, cols, q, g.pitch, s, qt, qt ? g.pitch_t : rows, st, fmt, limit, column_partial,
                   r.scale_format(), stream);
}

Tensor as_matrix(const Tensor& t, int64_t cols) {
    const Tensor flat = t.dim() == 2 ? t : t.reshape({-1, cols});
    TORCH_CHECK(flat.size(1) == cols, "expected ", cols, " features, got ", flat.size(1));
    return flat.is_contiguous() ? flat : flat.contiguous();
}

// Codes of the weight as the forward GEMM reads them: the stored ones, or for 16-bit storage freshly made; repacked where
// the rows are not whole pieces.
struct WeightSpace {
    int64_t q = -1, s = -1, p = -1, ps = -1, pitch = 0;
};

WeightSpace reserve_weight(const Layer& l, Arena& temp, int64_t pitch) {
    const Recipe& r = *l.recipe;
    WeightSpace w;
    w.pitch = pitch;
    const int64_t scale_rows = ceil_div(r.out, 32);
    if (!r.fp8_weight) {
        w.q = temp.take(r.out * r.in);
        w.s = temp.take(r.grouped ? scale_rows * ceil_div(r.in, 32) * r.scale_bytes() : 4);
    }
    if (w.pitch != r.in) {
        w.p = temp.take(r.out * w.pitch);
        if (r.grouped) w.ps = temp.take(scale_rows * ceil_div(w.pitch, 32) * r.scale_bytes());
    }
    return w;
}

// `scale_out` (per-tensor recipes with 16-bit storage): where the weight's scale goes instead of the arena
Codes stored_weight(const Layer& l, const Tensor& weight, const WeightSpace& w, const Arena& temp, float* scale_out, Codes* unpadded, viola_stream_t stream) {
    const Recipe& r = *l.recipe;
    Codes c{ptr(weight), ptr(l.scale), r.in};
    if (!r.fp8_weight) {
        const int dtype = code_of(weight.scalar_type());
        if (r.grouped) {
            c = {temp.at(w.q), temp.at(w.s), r.in};
            VIOLA_CALL(viola_group_quantize, ptr(weight), dtype, r.out, r.in, temp.at(w.q), r.fwd, temp.at(w.s), 32, 32, r.fwd_limit, 0, nullptr, 1, 32,
                       r.scale_format(), stream);
        } else {
            // a temporary workspace of block maxima
            Arena maxima;
            const int64_t at = maxima.take(1024 * 4);
            maxima.make(weight.device());
            c = {temp.at(w.q), scale_out, r.in};
            const Tensor& history = l.history[WEIGHT];
            VIOLA_CALL(viola_tensor_encode, ptr(weight), dtype, r.out, r.in, maxima.as<float>(at), 1024, static_cast<float*>(history.mutable_data_ptr()),
                       (int)history.numel(), l.counter[WEIGHT]->value, l.counter[WEIGHT]->delayed, r.fwd_limit, scale_out, temp.at(w.q), r.in, nullptr, 0, r.fwd, nullptr,
                       VIOLA_F32, stream);
            ++l.counter[WEIGHT]->value;
        }
    }
    if (unpadded) *unpadded = c;
    if (w.pitch != r.in) {
        void* scale_to = r.grouped ? temp.at(w.ps) : nullptr;
        VIOLA_CALL(viola_codes_repack, c.q, temp.at(w.p), 1, r.out, r.in, w.pitch, r.grouped ? c.s : nullptr, scale_to, 32, 32, r.scale_format(), stream);
        c = {temp.at(w.p), r.grouped ? scale_to : c.s, w.pitch};
    }
    return c;
}

// ---------------------------------------------------------------------------------------------------- one projection
// gated < 0: y = x W^T + b. gated >= 0 (an activation): y = act(g) * u of [g | u] = x W^T + b, and *aux = [g | u] when kept.
// hidden_out: (gated, grouped recipes) hand y over as codes instead of values where a kernel does; coded_input: x arrives that way.
struct CodedHidden {
    const Recipe* reader = nullptr;                              // the down projection's
    bool transposed = false;                                     // its weight gradient wants the other layout too
    Arena temp;                                                  // row-wise codes, used by this forward only
    Codes codes;                                                 // the other layout goes to the down projection's Kept arena
};

struct Forward {
    Tensor y, aux;
};

// The type of a parameter's gradient. A tensor that was itself computed (a parametrized weight) has no gradient type of its own.
at::ScalarType gradient_type(const Tensor& p) { return (p.is_leaf() ? p.grad_dtype() : std::nullopt).value_or(p.scalar_type()); }

Forward project(const Layer& l, const Tensor& x2, at::ScalarType dtype, bool need_backward, bool needs_w, Kept& kept, int gated, bool keep_aux,
                CodedHidden* hidden_out, Kept* hidden_kept, const CodedHidden* coded_input) {
    const Recipe& r = *l.recipe;
    const bool save = need_backward && needs_w;
    const int64_t rows = coded_input ? kept.rows : x2.size(0);
    const at::Device device = l.weight.device();
    const viola_stream_t stream = stream_of(l.weight);
    kept.rows = rows;
    kept.x_dtype = dtype;
    kept.has_input = save;
    if (need_backward) {
        kept.weight_t = l.transpose;
        kept.weight_t_scale = l.transpose_scale;
        kept.weight_grad = gradient_type(l.weight);
        if (l.bias.defined()) kept.bias_grad = gradient_type(l.bias);
    }
    const Tensor bias = l.bias.defined() ? l.bias.contiguous() : Tensor();      // the layer's own stays what the graph is connected to
    const auto options = at::TensorOptions().dtype(dtype).device(device);
    const int64_t h = r.out / 2;
    Forward f;
    if (rows == 0) {
        f.y = at::empty({0, gated < 0 ? r.out : h}, options);
        if (gated >= 0 && keep_aux) f.aux = at::empty({0, r.out}, options);
        return f;
    }
    Arena temp;
    const bool cache_here = !r.fp8_weight && need_backward && r.cache_transpose;   // 16-bit storage: W^T of this forward's codes
    // gated: through [g | u] by the plain product, where it is kept for backward anyway or the product is a small one
    const bool through_z = gated >= 0 && (keep_aux || (hidden_out && small_product(rows, r.out)));
    const bool plain = gated < 0 || (hidden_out && through_z && dtype != at::kFloat && h % 8 == 0);
    if (through_z) f.aux = at::empty({rows, r.out}, options);
    if (gated < 0) f.y = at::empty({rows, r.out}, options);
    Tensor& output = gated < 0 ? f.y : f.aux;
    // Nothing kept for backward and a small product: x is quantized inside it.
    auto quantized_inside = [&] {
        if (!plain || need_backward || coded_input || !r.fp8_weight || x2.element_size() != 2 || !small_product(rows, r.out)) return false;
        if ((rows > 16 && rows * r.out > 256 * 16 * 32 ? 2 : 1) * r.in > QUANTIZED_IN_PRODUCT) return false;
        if (!r.grouped && (rows * r.in > WHOLE_TENSOR || (l.counter[INPUT]->delayed && l.counter[INPUT]->value))) return false;
        const void* bias_p = ptr(bias);
        float* history = r.grouped ? nullptr : static_cast<float*>(l.history[INPUT].mutable_data_ptr());
        const int64_t slot = r.grouped ? 0 : l.counter[INPUT]->value % l.history[INPUT].numel();
        const int status = VIOLA_TRY(viola_skinny_linear, ptr(x2), code_of(x2.scalar_type()), nullptr, rows, r.in, ptr(l.weight), r.fwd, ptr(l.scale), r.grouped,
                                     r.out, r.fwd_limit, r.scale_format(), history, slot, nullptr, bias_p, bias_p ? code_of(bias.scalar_type()) : 0,
                                     output.mutable_data_ptr(), code_of(dtype), stream);
        if (status != 0 && status != VIOLA_EUNSUPPORTED) check("viola_skinny_linear", status);
        if (status == 0 && !r.grouped) ++l.counter[INPUT]->value;
        return status == 0;
    };
    const bool done = quantized_inside();
    if (done && gated < 0) return f;
    const int64_t pitch = plain ? product_pitch(r, rows, r.out, r.in) : r.pitch(r.in);
    Codes a, w, w_unpadded;
    if (!done) {
        const WeightSpace wspace = reserve_weight(l, temp, pitch);
        if (r.grouped) {
            GroupSpace g;
            if (!coded_input) g.reserve(r, &temp, save ? &kept.arena : nullptr, rows, r.in, pitch);
            temp.make(device);
            if (save && !coded_input) kept.arena.make(device);
            if (coded_input) {
                a = coded_input->codes;
            } else {
                Codes in_arena;
                quantize_groups(r, x2, r.fwd, r.fwd_limit, g, &temp, &kept.arena, nullptr, &a, &in_arena, stream);
                if (save) kept.input = {g.qt, g.st, g.pitch_t};
            }
            w = stored_weight(l, l.weight, wspace, temp, nullptr, &w_unpadded, stream);
        } else {
            const int64_t pitch_t = ceil_to(rows, 128);
            const int64_t q = temp.take(rows * pitch), maxima = temp.take(1024 * 4);
            const int64_t qt = save ? kept.arena.take(r.in * pitch_t) : -1;
            const int64_t scales = kept.arena.take(8);               // of x and of a 16-bit weight: backward uses these very values
            temp.make(device);
            kept.arena.make(device);
            float* sx = kept.arena.as<float>(scales);
            const Tensor& history = l.history[INPUT];
            VIOLA_CALL(viola_tensor_encode, ptr(x2), code_of(x2.scalar_type()), rows, r.in, temp.as<float>(maxima), 1024,
                       static_cast<float*>(history.mutable_data_ptr()), (int)history.numel(), l.counter[INPUT]->value, l.counter[INPUT]->delayed, r.fwd_limit, sx, temp.at(q),
                       pitch, save ? kept.arena.at(qt) : nullptr, save ? pitch_t : 0, r.fwd, nullptr, VIOLA_F32, stream);
            ++l.counter[INPUT]->value;
            a = {temp.at(q), sx, pitch};
            kept.scales = scales;
            if (save) kept.input = {qt, scales, pitch_t};
            w = stored_weight(l, l.weight, wspace, temp, sx + 1, &w_unpadded, stream);
        }
        if (cache_here) {
            kept.weight_t = at::empty({r.in, r.out}, at::TensorOptions().dtype(r.codes()).device(device));
            const bool grid = r.grouped;
            if (grid) kept.weight_t_scale = at::empty({ceil_div(r.in, 32), ceil_div(r.out, 32)}, at::TensorOptions().dtype(r.scales()).device(device));
            VIOLA_CALL(viola_codes_transpose_pitched, w_unpadded.q, kept.weight_t.mutable_data_ptr(), 1, r.out, r.in, r.out, grid ? w_unpadded.s : nullptr,
                       grid ? kept.weight_t_scale.mutable_data_ptr() : nullptr, 32, 32, r.scale_format(), nullptr, 0, 0, nullptr, 0, stream);
        }
        if (plain) product(r, a, r.fwd, w, r.fwd, rows, r.out, 32, bias, output.mutable_data_ptr(), dtype, device, stream);
    }
    if (gated < 0) return f;
    if (plain) {
        // one pass over [g | u] makes h's codes; h itself is never stored
        const Recipe& to = *hidden_out->reader;
        GroupSpace space;
        space.reserve(to, &hidden_out->temp, hidden_out->transposed ? &hidden_kept->arena : nullptr, rows, h, product_pitch(to, rows, to.out, h));
        hidden_out->temp.make(device);
        hidden_kept->arena.make(device);
        hidden_out->codes = {hidden_out->temp.at(space.q), hidden_out->temp.at(space.s), space.pitch};
        if (hidden_out->transposed) hidden_kept->input = {space.qt, space.st, space.pitch_t};
        VIOLA_CALL(viola_gated_quantize_dual_pitched, ptr(f.aux), code_of(dtype), rows, h, gated, const_cast<void*>(hidden_out->codes.q), space.pitch,
                   const_cast<void*>(hidden_out->codes.s), hidden_out->transposed ? hidden_kept->arena.at(space.qt) : nullptr,
                   hidden_out->transposed ? space.pitch_t : rows, hidden_out->transposed ? hidden_kept->arena.at(space.st) : nullptr, to.fwd, to.fwd_limit,
                   to.scale_format(), stream);
        hidden_kept->rows = rows;
        return f;
    }
    // whole 128 x 128 pieces in both directions: the codes need no padding on either k axis of the down projection
    if (hidden_out && r.native && rows % 128 == 0 && h % 128 == 0) {
        // h leaves the product as codes with E8M0 scales in the layouts the down projection reads (its k is h wide)
        const bool transposed = hidden_out->transposed;
        Arena& keep = hidden_kept->arena;
        const int64_t q = hidden_out->temp.take(rows * h), s = hidden_out->temp.take(rows * (h / 32));
        const int64_t qt = transposed ? keep.take(h * rows) : -1, st = transposed ? keep.take(h * (rows / 32)) : -1;
        hidden_out->temp.make(device);
        keep.make(device);
        void* qt_p = transposed ? keep.at(qt) : nullptr;
        uint8_t* st_p = transposed ? keep.as<uint8_t>(st) : nullptr;
        const void* bias_p = ptr(bias);
        const int status = VIOLA_TRY(viola_mx_gated_gemm_encode, a.q, r.fwd, w.q, r.fwd, static_cast<const uint8_t*>(a.s), static_cast<const uint8_t*>(w.s), rows, h,
                                     a.pitch, 1, 32, bias_p, bias_p ? code_of(bias.scalar_type()) : 0, const_cast<void*>(ptr(f.aux)), code_of(dtype),
                                     hidden_out->temp.at(q), hidden_out->temp.as<uint8_t>(s), qt_p, st_p, r.fwd, r.fwd_limit, gated, stream);
        if (status != 0 && status != VIOLA_EUNSUPPORTED) check("viola_mx_gated_gemm_encode", status);
        if (status == 0) {
            hidden_out->codes = {hidden_out->temp.at(q), hidden_out->temp.at(s), h};
            if (transposed) hidden_kept->input = {qt, st, rows};
            hidden_kept->rows = rows;
            return f;
        }
        hidden_kept->arena = Arena();
    }
    f.y = at::empty({rows, h}, options);
    gated_product(r, a, r.fwd, w, r.fwd, rows, h, bias, f.aux, f.y, gated, false, stream);
    return f;
}

struct Gradients {
    Tensor dx, dw, db;
};

// The up projection's dy is dz of this [g | u] and of the dh handed over as dy.
struct GatedGradient {
    Tensor z;
    int activation = 0;
};

// gated >= 0: dx is dz = [d u act'(g) | d act(g)] from aux = [g | u].
Gradients unproject(const Layer& l, const Kept& kept, const Restored& t, const Tensor& dy_, bool needs_x, bool needs_w, bool needs_b, int gated, const Tensor& aux,
                    const GatedGradient* gate = nullptr) {
    const Recipe& r = *l.recipe;
    const int64_t rows = kept.rows;
    const Tensor& w = t.weight;
    const at::Device device = w.device();
    const viola_stream_t stream = stream_of(w);
    const auto dx_options = at::TensorOptions().dtype(kept.x_dtype).device(device);
    const int64_t dx_cols = gated < 0 ? r.in : 2 * r.in;
    Gradients out;
    if (rows == 0) {
        if (needs_x) out.dx = at::zeros({0, dx_cols}, dx_options);
        if (needs_w) out.dw = at::zeros({r.out, r.in}, dx_options.dtype(kept.weight_grad));
        if (needs_b) out.db = at::zeros({r.out}, dx_options.dtype(kept.bias_grad));
        return out;
    }
    const Tensor dy = as_matrix(dy_, gate ? r.out / 2 : r.out);
    Arena temp;
    Codes g, gt, wt;
    float* partial = nullptr;
    const int64_t parts = ceil_div(rows, 32), pitch = gated < 0 ? product_pitch(r, rows, r.in, r.out) : r.pitch(r.out);
    // ---- space for the transposed weight
    const bool cached = kept.has_weight_t;
    const bool make_wt = needs_x && !(cached && pitch == r.out);
    const int64_t wt_q = make_wt ? temp.take(r.in * pitch) : -1, wt_s = make_wt && r.grouped ? temp.take(ceil_div(r.in, 32) * ceil_div(pitch, 32) * r.scale_bytes()) : -1;
    const bool requantize = make_wt && !cached && !r.fp8_weight; // memory mode with 16-bit storage: this forward's codes again
    const int64_t w_q = requantize ? temp.take(r.out * r.in) : -1;
    const int64_t w_s = requantize && r.grouped ? temp.take(ceil_div(r.out, 32) * ceil_div(r.in, 32) * r.scale_bytes()) : -1;
    // per-tensor codes as stored: the quantizer of dy turns them in its own launch where they are whole words
    const bool beside = make_wt && !cached && !requantize && !r.grouped && r.out % 4 == 0 && r.in % 4 == 0 && pitch % 4 == 0 && reinterpret_cast<uintptr_t>(ptr(w)) % 4 == 0;
    if (needs_b) out.db = at::empty({r.out}, dx_options.dtype(kept.bias_grad));
    int k_parts = 1;                                             // of the weight gradient's k range, and the partial products
    int64_t k_parts_at = -1;
    if (r.grouped) {
        GroupSpace space;
        space.reserve(r, needs_x ? &temp : nullptr, needs_w ? &temp : nullptr, rows, r.out, pitch);
        const int64_t size = r.out * r.in;
        if (needs_w && !r.native) k_parts = viola_group_gemm_parts(r.out, r.in, space.pitch_t);
        if (k_parts > 1) k_parts_at = temp.take(k_parts * ceil_to(size, 4) * 4);
        const bool rides = needs_b && needs_w;                   // the bias gradient's 32-row sums come from the quantizer's read of dy
        const int64_t partial_at = rides ? temp.take(parts * r.out * 4) : -1;
        temp.make(device);
        if (rides) partial = temp.as<float>(partial_at);
        if (gate) {
            void *q = nullptr, *s = nullptr, *qt = nullptr, *st = nullptr;
            if (needs_x) { q = temp.at(space.q); s = temp.at(space.s); g = {q, s, space.pitch}; }
            if (needs_w) { qt = temp.at(space.qt); st = temp.at(space.st); gt = {qt, st, space.pitch_t}; }
            VIOLA_CALL(viola_gated_backward_quantize_dual, ptr(gate->z), ptr(dy), code_of(dy.scalar_type()), rows, r.out / 2, gate->activation, q, s, qt,
                       needs_w ? space.pitch_t : rows, st, r.bwd, r.bwd_limit, partial, r.scale_format(), stream);
        } else if (needs_x || needs_w) quantize_groups(r, dy, r.bwd, r.bwd_limit, space, &temp, &temp, partial, &g, &gt, stream);
        if (needs_b && !rides) out.db = at::sum(dy, at::IntArrayRef{0}, false, kept.bias_grad);
    } else {
        const int64_t pitch_t = ceil_to(rows, 128);
        const int64_t q = needs_x ? temp.take(rows * pitch) : -1, qt = needs_w ? temp.take(r.out * pitch_t) : -1, scale_at = temp.take(4);
        const int dtype = code_of(dy.scalar_type());
        bool rides = needs_b;
        const int64_t floats = 1024 + (rides ? viola_tensor_encode_slices(dtype, rows, r.out) * r.out : 0), work_at = temp.take(floats * 4);
        temp.make(device);
        float* scale = temp.as<float>(scale_at);
        const Tensor& history = l.history[GRAD];
        auto encode = [&](bool with_sum) {
            return VIOLA_TRY(viola_tensor_encode_beside, ptr(dy), dtype, rows, r.out, temp.as<float>(work_at), floats, static_cast<float*>(history.mutable_data_ptr()),
                             (int)history.numel(), l.counter[GRAD]->value, l.counter[GRAD]->delayed, r.bwd_limit, scale, needs_x ? temp.at(q) : nullptr, pitch,
                             needs_w ? temp.at(qt) : nullptr, pitch_t, r.bwd, with_sum ? out.db.mutable_data_ptr() : nullptr,
                             with_sum ? code_of(kept.bias_grad) : VIOLA_F32, beside ? ptr(w) : nullptr, beside ? temp.at(wt_q) : nullptr, r.out, r.in, pitch,
                             stream);
        };
        int status = encode(rides);
        if (status == VIOLA_EUNSUPPORTED && rides) {             // columns that are not whole 16-byte pieces: the sum as a pass of its own
            out.db = at::sum(dy, at::IntArrayRef{0}, false, kept.bias_grad);
            status = encode(false);
        }
        check("viola_tensor_encode_beside", status);
        ++l.counter[GRAD]->value;
        if (needs_x) g = {temp.at(q), scale, pitch};
        if (needs_w) gt = {temp.at(qt), scale, pitch_t};
    }
    if (needs_x) {
        const void* w_scale = r.fp8_weight ? ptr(t.weight_scale) : r.grouped ? nullptr : t.scales + 1;
        wt = {ptr(t.weight_t), r.grouped ? ptr(t.weight_t_scale) : w_scale, pitch};
        if (make_wt && cached) {
            VIOLA_CALL(viola_codes_repack, ptr(t.weight_t), temp.at(wt_q), 1, r.in, r.out, pitch, r.grouped ? ptr(t.weight_t_scale) : nullptr,
                       r.grouped ? temp.at(wt_s) : nullptr, 32, 32, r.scale_format(), stream);
        } else if (make_wt && !beside) {
            const void* codes = ptr(w);
            if (requantize) {
                codes = temp.at(w_q);
                if (r.grouped) {
                    w_scale = temp.at(w_s);
                    VIOLA_CALL(viola_group_quantize, ptr(w), code_of(w.scalar_type()), r.out, r.in, temp.at(w_q), r.fwd, temp.at(w_s), 32, 32, r.fwd_limit, 0,
                               nullptr, 1, 32, r.scale_format(), stream);
                } else {
                    VIOLA_CALL(viola_tensor_quantize, ptr(w), code_of(w.scalar_type()), r.out, r.in, static_cast<const float*>(w_scale), temp.at(w_q), nullptr,
                               r.fwd, r.fwd_limit, stream);
                }
            }
            VIOLA_CALL(viola_codes_transpose_pitched, codes, temp.at(wt_q), 1, r.out, r.in, pitch, r.grouped ? w_scale : nullptr,
                       r.grouped ? temp.at(wt_s) : nullptr, 32, 32, r.scale_format(), partial, parts, r.out, partial ? out.db.mutable_data_ptr() : nullptr,
                       partial ? code_of(kept.bias_grad) : VIOLA_F32, stream);
            partial = nullptr;                                   // reduced by the same launch
        }
        if (make_wt) wt = {temp.at(wt_q), r.grouped ? temp.at(wt_s) : w_scale, pitch};
    }
    if (partial) VIOLA_CALL(viola_column_reduce, partial, parts, r.out, out.db.mutable_data_ptr(), code_of(kept.bias_grad), stream);
    if (needs_x) {
        out.dx = at::empty({rows, dx_cols}, dx_options);
        if (gated < 0) product(r, g, r.bwd, wt, r.fwd, rows, r.in, 32, Tensor(), out.dx.mutable_data_ptr(), kept.x_dtype, device, stream);
        else gated_product(r, g, r.bwd, wt, r.fwd, rows, r.in, Tensor(), aux, out.dx, gated, true, stream);
    }
    if (needs_w) {
        out.dw = at::empty({r.out, r.in}, dx_options.dtype(kept.weight_grad));
        int status = VIOLA_EUNSUPPORTED;
        if (k_parts > 1) {
            TORCH_INTERNAL_ASSERT(gt.pitch == t.input_t.pitch);
            status = VIOLA_TRY(viola_group_gemm_in_parts, gt.q, r.bwd, t.input_t.q, r.fwd, static_cast<const float*>(gt.s), static_cast<const float*>(t.input_t.s),
                               r.out, r.in, gt.pitch, out.dw.mutable_data_ptr(), code_of(kept.weight_grad), k_parts, temp.as<float>(k_parts_at),
                               k_parts * ceil_to(r.out * r.in, 4), stream);
            if (status != VIOLA_EUNSUPPORTED) check("viola_group_gemm_in_parts", status);
        }
        if (status != 0) product(r, gt, r.bwd, t.input_t, r.fwd, r.out, r.in, 1, Tensor(), out.dw.mutable_data_ptr(), kept.weight_grad, device, stream);
    }
    return out;
}

// The two projections of an MLP hand h over in one form: one of them replaced by a Linear of another recipe is the general path's.
bool pair(const Recipe& up, const Recipe& down) {
    return up.out == 2 * down.in && up.grouped == down.grouped && up.native == down.native && up.fwd == down.fwd && up.fwd_limit == down.fwd_limit;
}

bool wants(const Tensor& t) { return t.defined() && t.requires_grad(); }

// ---------------------------------------------------------------------------------------------------- Linear
struct LinearBackward : public Node {
    Layer layer;                                                 // without its tensors, but for the quantizers' histories
    Kept kept;
    std::vector<int64_t> x_shape;

    variable_list apply(variable_list&& grads) override {
        const Tensor& dy = grads[0];
        variable_list result(3);
        if (!dy.defined()) return result;
        const Restored tensors = restore(kept, *layer.recipe, dy);
        at::AutoDispatchBelowADInplaceOrView below;
        Gradients g = unproject(layer, kept, tensors, dy, task_should_compute_output(0), task_should_compute_output(1) && kept.has_input,
                                task_should_compute_output(2), -1, Tensor());
        if (g.dx.defined()) result[0] = g.dx.dim() == (int64_t)x_shape.size() ? g.dx : g.dx.view(x_shape);
        result[1] = g.dw;
        result[2] = g.db;
        return result;
    }
    std::string name() const override { return "ViolaLinearBackward"; }
    void release_variables() override { kept.release(); }
};

std::vector<int64_t> output_shape(const Tensor& x, int64_t features) {
    std::vector<int64_t> shape = x.sizes().vec();
    shape.back() = features;
    return shape;
}

// The histories are updated in place by raw pointers; nothing else of the layer's tensors is kept by a node.
Layer without_tensors(const Layer& l) {
    Layer kept;
    kept.recipe = l.recipe;
    for (int i = 0; i < 3; ++i) { kept.history[i] = l.history[i]; kept.counter[i] = l.counter[i]; }
    return kept;
}

Tensor linear(const Tensor& x, Layer& l) {
    const bool wx = x.requires_grad(), ww = l.weight.requires_grad(), wb = wants(l.bias);
    const bool need = at::GradMode::is_enabled() && (wx || ww || wb);
    auto node = need ? std::shared_ptr<LinearBackward>(new LinearBackward(), torch::autograd::deleteNode) : nullptr;
    Kept scratch;
    Kept& kept = need ? node->kept : scratch;
    Tensor y;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor x2 = as_matrix(x, l.recipe->in);
        y = project(l, x2, x.scalar_type(), need, ww, kept, -1, false, nullptr, nullptr, nullptr).y;
        if (x.dim() != 2) y = y.view(output_shape(x, l.recipe->out));
    }
    if (need) {
        node->layer = without_tensors(l);
        node->kept.save(l);
        node->x_shape = x.sizes().vec();
        node->set_next_edges(torch::autograd::collect_next_edges(x, l.weight, l.bias));
        torch::autograd::set_history(y, node);
    }
    return y;
}

// ---------------------------------------------------------------------------------------------------- MLP
// One node for the whole gated MLP. Grouped and block-scaled recipes: the down projection's data-gradient product writes dh, and
// the quantizer of the stacked gate/up projection's gradient makes dz, the gradient of [g | u], as it reads dh and [g | u]; dz is
// never stored. Per-tensor recipes, whose scale needs dz before it is quantized, and shapes that quantizer does not take: the
// product itself hands out dz (viola_*_gated_gemm: in its epilogue, or on large tiles in one pass over dh).
struct MlpBackward : public Node {
    Layer up, down;
    Kept up_kept, down_kept;
    SavedVariable z;
    std::vector<int64_t> x_shape;
    int activation = 0;
    bool first_half = false;

    variable_list apply(variable_list&& grads) override {
        const Tensor& dy = grads[0];
        variable_list result(5);
        if (!dy.defined()) return result;
        const Restored down_tensors = restore(down_kept, *down.recipe, dy);
        const bool upper = first_half && (task_should_compute_output(0) || task_should_compute_output(1) || task_should_compute_output(2));
        const bool up_x = task_should_compute_output(0), up_w = task_should_compute_output(1) && up_kept.has_input, up_b = task_should_compute_output(2);
        // grouped recipes: the plain product writes dh, and the quantizer of dz makes dz as it reads dh and [g | u]
        const bool direct = upper && up.recipe->grouped && up_kept.rows && up_kept.x_dtype != at::kFloat && down.recipe->in % 64 == 0 && (up_w || (up_x && !up_b));
        const Restored up_tensors = upper ? restore(up_kept, *up.recipe, dy) : Restored();
        GatedGradient gate{upper ? restored(z, dy.device(), up_kept.x_dtype, {up_kept.rows, up.recipe->out}) : Tensor(), activation};
        at::AutoDispatchBelowADInplaceOrView below;
        Gradients d = unproject(down, down_kept, down_tensors, dy, upper, task_should_compute_output(3) && down_kept.has_input, task_should_compute_output(4),
                                direct ? -1 : activation, gate.z);
        result[3] = d.dw;
        result[4] = d.db;
        if (!upper) return result;
        Gradients u = unproject(up, up_kept, up_tensors, d.dx, up_x, up_w, up_b, -1, Tensor(), direct ? &gate : nullptr);
        if (u.dx.defined()) result[0] = u.dx.dim() == (int64_t)x_shape.size() ? u.dx : u.dx.view(x_shape);
        result[1] = u.dw;
        result[2] = u.db;
        return result;
    }
    std::string name() const override { return "ViolaMLPBackward"; }
    void release_variables() override {
        up_kept.release();
        down_kept.release();
        z.reset_data();
    }
};

Tensor mlp(const Tensor& x, Layer& up, Layer& down, int activation) {
    const bool grad = at::GradMode::is_enabled();
    const bool up_w = up.weight.requires_grad(), down_w = down.weight.requires_grad();
    const bool first_half = grad && (x.requires_grad() || up_w || wants(up.bias));
    const bool whole = grad && (first_half || down_w || wants(down.bias));
    auto node = whole ? std::shared_ptr<MlpBackward>(new MlpBackward(), torch::autograd::deleteNode) : nullptr;
    Kept scratch_up, scratch_down;
    Kept& up_kept = whole ? node->up_kept : scratch_up;
    Kept& down_kept = whole ? node->down_kept : scratch_down;
    Tensor y, z;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor x2 = as_matrix(x, up.recipe->in);
        const int64_t rows = x2.size(0);
        CodedHidden hidden;
        hidden.reader = down.recipe.get();
        hidden.transposed = whole && down_w;
        const bool as_codes = up.recipe->grouped && rows > 0;
        Forward first = project(up, x2, x.scalar_type(), first_half, up_w, up_kept, activation, first_half, as_codes ? &hidden : nullptr,
                                as_codes ? &down_kept : nullptr, nullptr);
        z = first.aux;
        const bool coded = !first.y.defined();
        y = project(down, first.y, x.scalar_type(), whole, down_w, down_kept, -1, false, nullptr, nullptr, coded ? &hidden : nullptr).y;
        if (x.dim() != 2) y = y.view(output_shape(x, down.recipe->out));
    }
    if (whole) {
        node->up = without_tensors(up);
        node->down = without_tensors(down);
        node->activation = activation;
        node->first_half = first_half;
        node->x_shape = x.sizes().vec();
        if (first_half) {
            node->up_kept.save(up);
            node->z = SavedVariable(z, false);
        } else {
            node->up_kept.arena.release();
        }
        node->down_kept.save(down);
        node->set_next_edges(torch::autograd::collect_next_edges(x, up.weight, up.bias, down.weight, down.bias));
        torch::autograd::set_history(y, node);
    }
    return y;
}

// ---------------------------------------------------------------------------------------------------- variable groups
struct Groups {
    int64_t count = 0, rows = 0, padded = 0;
    Arena arena;                                                 // forward only: row offsets, then offsets on the padded token axis
    const int64_t* offsets = nullptr;
    const int64_t* padded_offsets = nullptr;
    void at(const Tensor& table) {
        offsets = static_cast<const int64_t*>(table.const_data_ptr());
        padded_offsets = offsets + count + 1;
    }
};

// The offset tables travel as kernel arguments: no staging buffer, no copy the host has to wait for.
void make_groups(Groups& g, const std::vector<int64_t>& counts, const at::Device& device, viola_stream_t stream) {
    g.count = (int64_t)counts.size();
    std::vector<int64_t> words(2 * (g.count + 1), 0);
    int64_t* padded = words.data() + g.count + 1;
    for (int64_t i = 0; i < g.count; ++i) {
        TORCH_CHECK(counts[i] >= 0, "rows per group cannot be negative");
        words[i + 1] = words[i] + counts[i];
        padded[i + 1] = padded[i] + ceil_to(counts[i], 32);
    }
    // The padded token axis is the row length of the transposed codes: rounded up to 128 (empty slots at the end of the last
    // group, zero codes) so that every row starts on a cache line and the quantizer's 64-byte pieces never straddle one.
    padded[g.count] = ceil_to(padded[g.count], 128);
    g.rows = words[g.count];
    g.padded = padded[g.count];
    const int64_t at = g.arena.take((int64_t)words.size() * 8);
    g.arena.make(device);
    VIOLA_CALL(viola_store_words, g.arena.as<int64_t>(at), words.data(), (int64_t)words.size(), stream);
    g.at(g.arena.tensor());
}

struct ExpertsBackward : public Node {
    std::shared_ptr<Recipe> recipe;
    Groups groups;
    Arena kept;                                                  // forward only: transposed codes of x
    Place input;                                                 // in the saved arena
    SavedVariable tables, saved_arena, weight, weight_scale;     // see Kept
    std::vector<int64_t> weight_shape;
    int weight_fmt = VIOLA_E4M3;
    at::ScalarType x_dtype = at::kFloat, weight_grad = at::kFloat;
    bool has_input = false;

    variable_list apply(variable_list&& grads) override;
    std::string name() const override { return "ViolaExpertsBackward"; }
    void release_variables() override {
        for (SavedVariable* v : {&tables, &saved_arena, &weight, &weight_scale}) v->reset_data();
    }
};

// x's row-wise codes and, where asked for, its per-group transposed codes; one read of x where the kernel takes the shape
void quantize_segments(const Recipe& r, const Tensor& x, int fmt, float limit, const Groups& g, const Arena* rowwise, const GroupSpace& space, void* qt,
                       float* st, Codes* out, viola_stream_t stream) {
    const int64_t rows = x.size(0), cols = x.size(1);
    const int dtype = code_of(x.scalar_type());
    const bool together = qt && rowwise && x.element_size() == 2 && cols % 8 == 0 && space.pitch == cols && reinterpret_cast<uintptr_t>(ptr(x)) % 16 == 0;
    if (qt)
        VIOLA_CALL(viola_varlen_quantize_transposed, ptr(x), dtype, rows, cols, g.offsets, g.padded_offsets, (int)g.count, g.padded, qt, st, fmt, limit,
                   together ? rowwise->at(space.q) : nullptr, together ? rowwise->as<float>(space.s) : nullptr, stream);
    if (!rowwise) return;
    Codes unused;
    if (together) *out = {rowwise->at(space.q), rowwise->at(space.s), space.pitch};
    else quantize_groups(r, x, fmt, limit, space, rowwise, nullptr, nullptr, out, &unused, stream);
}

void segment_product(const Recipe& r, const Codes& a, int a_fmt, const Codes& b, int b_fmt, const Groups& g, int64_t n, void* out, at::ScalarType dtype,
                     viola_stream_t stream) {
    const int64_t k = a.pitch;
    VIOLA_CALL(viola_varlen_group_gemm, a.q, a_fmt, b.q, b_fmt, static_cast<const float*>(a.s), static_cast<const float*>(b.s), g.offsets, (int)g.count, g.rows,
               n, k, 1, 32, 32, 32, n * k, ceil_div(n, 32) * ceil_div(k, 32), out, code_of(dtype), stream);
}

Tensor experts(const Tensor& x_, const Tensor& weight, const Tensor& weight_scale, const std::vector<int64_t>& counts, const std::shared_ptr<Recipe>& recipe,
               at::ScalarType weight_grad) {
    TORCH_CHECK(x_.is_cuda() && x_.dim() == 2 && weight.dim() == 3 && weight.size(0) == (int64_t)counts.size() && x_.size(1) == weight.size(2));
    const int w_fmt = code_of(weight.scalar_type());             // the codes' own format, whatever the recipe encodes x in
    TORCH_CHECK((w_fmt == VIOLA_E4M3 || w_fmt == VIOLA_E5M2) && weight.is_contiguous() && weight.device() == x_.device(), "weight: contiguous FP8 codes on x's device");
    TORCH_CHECK(holds(weight_scale, x_.device(), at::kFloat, {weight.size(0), ceil_div(weight.size(1), 32), ceil_div(weight.size(2), 32)}),
                "weight_scale: contiguous FP32 [groups, ceil(out / 32), ceil(in / 32)] on x's device");
    const Recipe& r = *recipe;
    const bool wx = x_.requires_grad(), ww = weight.requires_grad();
    const bool need = at::GradMode::is_enabled() && (wx || ww);
    auto node = need ? std::shared_ptr<ExpertsBackward>(new ExpertsBackward(), torch::autograd::deleteNode) : nullptr;
    const int64_t n = weight.size(1), k = weight.size(2);
    Tensor y;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor x = x_.contiguous();
        const at::Device device = x.device();
        const viola_stream_t stream = stream_of(x);
        Groups scratch_groups;
        Groups& groups = need ? node->groups : scratch_groups;
        make_groups(groups, counts, device, stream);
        TORCH_CHECK(groups.rows == x.size(0), "the group sizes add up to ", groups.rows, " rows, x has ", x.size(0));
        const bool save = need && ww && groups.rows;
        Arena temp;
        GroupSpace space;
        space.reserve(r, &temp, nullptr, groups.rows, k, r.pitch(k));
        const bool repack = space.pitch != k;
        const int64_t wp = repack ? temp.take(groups.count * n * space.pitch) : -1;
        const int64_t wps = repack ? temp.take(groups.count * ceil_div(n, 32) * ceil_div(space.pitch, 32) * 4) : -1;
        temp.make(device);
        void* qt = nullptr;
        float* st = nullptr;
        if (save) {
            const int64_t q_at = node->kept.take(k * groups.padded), s_at = node->kept.take(k * (groups.padded / 32) * 4);
            node->kept.make(device);
            qt = node->kept.at(q_at);
            st = node->kept.as<float>(s_at);
            node->input = {q_at, s_at, groups.padded};
        }
        y = at::empty({groups.rows, n}, x.options());
        if (groups.rows) {
            Codes a, w{ptr(weight), ptr(weight_scale), k};
            quantize_segments(r, x, r.fwd, r.fwd_limit, groups, &temp, space, qt, st, &a, stream);
            if (repack) {
                VIOLA_CALL(viola_codes_repack, w.q, temp.at(wp), groups.count, n, k, space.pitch, w.s, temp.at(wps), 32, 32, VIOLA_SCALE_F32, stream);
                w = {temp.at(wp), temp.at(wps), space.pitch};
            }
            segment_product(r, a, r.fwd, w, w_fmt, groups, n, y.mutable_data_ptr(), x.scalar_type(), stream);
        }
        if (need) {
            node->has_input = save;
            node->x_dtype = x.scalar_type();
        }
    }
    if (need) {
        node->recipe = recipe;
        node->weight = SavedVariable(weight, false);
        node->weight_scale = SavedVariable(weight_scale, false);
        node->tables = SavedVariable(node->groups.arena.tensor(), false);
        node->saved_arena = SavedVariable(node->kept.tensor(), false);
        node->groups.arena.release();
        node->kept.release();
        node->weight_shape = weight.sizes().vec();
        node->weight_fmt = w_fmt;
        node->weight_grad = weight_grad;
        node->set_next_edges(torch::autograd::collect_next_edges(x_, weight));
        torch::autograd::set_history(y, node);
    }
    return y;
}

variable_list ExpertsBackward::apply(variable_list&& grads) {
    variable_list result(2);
    if (!grads[0].defined()) return result;
    const Recipe& r = *recipe;
    const Tensor w = weight.unpack().contiguous();
    TORCH_CHECK(w.device() == grads[0].device() && w.sizes() == at::IntArrayRef(weight_shape) && code_of(w.scalar_type()) == weight_fmt,
                "the weight of a grouped linear was moved or replaced between forward and backward");
    const int w_fmt = weight_fmt;
    const int64_t count = w.size(0), n = w.size(1), k = w.size(2);
    const Tensor scale = restored(weight_scale, w.device(), at::kFloat, {count, ceil_div(n, 32), ceil_div(k, 32)});
    const Tensor table = restored(tables, w.device(), at::kByte, {groups.arena.size()});
    const Tensor codes = has_input ? restored(saved_arena, w.device(), at::kByte, {kept.size()}) : Tensor();
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor dy = as_matrix(grads[0], n);
    Groups groups = this->groups;                                // a second backward pass may run beside this one
    groups.at(table);
    const at::Device device = w.device();
    const viola_stream_t stream = stream_of(w);
    const bool needs_x = task_should_compute_output(0), needs_w = task_should_compute_output(1);
    const auto options = at::TensorOptions().device(device);
    if (needs_w && !groups.rows) result[1] = at::zeros({count, n, k}, options.dtype(weight_grad));
    if (needs_x && !groups.rows) result[0] = at::empty({0, k}, options.dtype(x_dtype));
    if (!groups.rows) return result;
    const bool weight_too = needs_w && has_input;
    Arena temp;
    GroupSpace space;
    space.reserve(r, needs_x ? &temp : nullptr, nullptr, groups.rows, n, r.pitch(n));
    const int64_t scale_cols = ceil_div(space.pitch, 32);
    const int64_t wt = needs_x ? temp.take(count * k * space.pitch) : -1, wts = needs_x ? temp.take(count * ceil_div(k, 32) * scale_cols * 4) : -1;
    const int64_t qt = weight_too ? temp.take(n * groups.padded) : -1, st = weight_too ? temp.take(n * (groups.padded / 32) * 4) : -1;
    temp.make(device);
    Codes g;
    quantize_segments(r, dy, r.bwd, r.bwd_limit, groups, needs_x ? &temp : nullptr, space, weight_too ? temp.at(qt) : nullptr,
                      weight_too ? temp.as<float>(st) : nullptr, &g, stream);
    if (needs_x) {
        VIOLA_CALL(viola_codes_transpose_pitched, ptr(w), temp.at(wt), count, n, k, space.pitch, ptr(scale), temp.at(wts), 32, 32, VIOLA_SCALE_F32, nullptr, 0,
                   0, nullptr, 0, stream);
        result[0] = at::empty({groups.rows, k}, options.dtype(x_dtype));
        segment_product(r, g, r.bwd, Codes{temp.at(wt), temp.at(wts), space.pitch}, w_fmt, groups, k, result[0].mutable_data_ptr(), x_dtype, stream);
    }
    if (weight_too) {
        result[1] = at::empty({count, n, k}, options.dtype(weight_grad));
        const Codes input_t = input.in(codes.const_data_ptr());
        VIOLA_CALL(viola_varlen_wgrad_gemm, temp.at(qt), r.bwd, input_t.q, r.fwd, temp.as<float>(st), static_cast<const float*>(input_t.s), groups.padded_offsets,
                   (int)count, groups.padded, n, k, result[1].mutable_data_ptr(), code_of(weight_grad), stream);
    }
    return result;
}

// quantize_segments as an operator of its own: (qt, st), with `rowwise` also the row-wise codes and scales (views of padded rows)
std::vector<Tensor> segments(const Tensor& x, const Recipe& r, const Tensor& offsets, const Tensor& padded_offsets, int64_t count, int64_t padded, bool rowwise) {
    TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous());
    const int64_t rows = x.size(0), cols = x.size(1);
    const at::Device device = x.device();
    for (const Tensor* t : {&offsets, &padded_offsets})
        TORCH_CHECK(holds(*t, device, at::kLong, {count + 1}), "offsets: contiguous int64 [groups + 1] on x's device");
    Groups g;
    g.count = count; g.rows = rows; g.padded = padded;
    g.offsets = offsets.const_data_ptr<int64_t>(); g.padded_offsets = padded_offsets.const_data_ptr<int64_t>();
    const auto options = at::TensorOptions().device(device);
    const Tensor qt = at::empty({cols, padded}, options.dtype(r.codes())), st = at::empty({cols, padded / 32}, options.dtype(at::kFloat));
    Arena temp;
    GroupSpace space;
    if (rowwise) space.reserve(r, &temp, nullptr, rows, cols, r.pitch(cols));
    temp.make(device);
    Codes out;
    quantize_segments(r, x, r.fwd, r.fwd_limit, g, rowwise ? &temp : nullptr, space, qt.mutable_data_ptr(), st.mutable_data_ptr<float>(), &out, stream_of(x));
    if (!rowwise) return {qt, st};
    const int64_t scales = ceil_div(space.pitch, 32);
    const Tensor q = temp.tensor().narrow(0, space.q, rows * space.pitch).view({rows, space.pitch}).view(r.codes());
    const Tensor s = temp.tensor().narrow(0, space.s, rows * scales * 4).view({rows, scales * 4}).view(at::kFloat);
    return {qt, st, q.narrow(1, 0, cols), s.narrow(1, 0, ceil_div(cols, 32))};
}

// ---------------------------------------------------------------------------------------------------- Python
// (recipe, weight, bias, scale, transpose, transpose scale[, three histories, three counters])
Layer layer_from(const py::tuple& t) {
    Layer l;
    l.recipe = t[0].cast<std::shared_ptr<Recipe>>();
    l.weight = t[1].cast<Tensor>();
    if (!t[2].is_none()) l.bias = t[2].cast<Tensor>();
    l.scale = t[3].cast<Tensor>();
    l.transpose = t[4].cast<Tensor>();
    l.transpose_scale = t[5].cast<Tensor>();
    if (t.size() > 6)
        for (int i = 0; i < 3; ++i) {
            l.history[i] = t[6 + i].cast<Tensor>();
            l.counter[i] = t[9 + i].cast<std::shared_ptr<Counter>>();
        }
    return l;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
    event_class = new py::object(py::module_::import("torch.cuda").attr("Event"));
    py::class_<Counter, std::shared_ptr<Counter>>(m, "Counter")
        .def(py::init([](int64_t value, bool delayed) { return std::make_shared<Counter>(value, delayed); }), py::arg("value") = 0, py::arg("delayed") = false)
        .def_property("value", [](const Counter& c) { return c.value.load(); }, [](Counter& c, int64_t value) { c.value = value; })
        .def_property("delayed", [](const Counter& c) { return c.delayed.load(); }, [](Counter& c, bool delayed) { c.delayed = delayed; })
        .def("__reduce__", [](py::object self) { return py::make_tuple(self.attr("__class__"), py::make_tuple(self.attr("value"), self.attr("delayed"))); });
    py::class_<Recipe, std::shared_ptr<Recipe>>(m, "Recipe")
        .def(py::init<const py::dict&>())
        .def("__reduce__", [](py::object self) { return py::make_tuple(self.attr("__class__"), py::make_tuple(self.cast<Recipe&>().fields())); });
    m.def("set_timeline", [](py::object list) {
        if (!timeline_sink) timeline_sink = new py::object();
        *timeline_sink = list;
        recording.store(!list.is_none());
    });
    register_optimizer(m);
    m.def("segment_offsets", torch::wrap_pybind_function([](const std::vector<int64_t>& counts, const at::Device& device) {
        Groups g;
        make_groups(g, counts, device, c10::hip::getCurrentHIPStream(device.index()).stream());
        return g.arena.tensor();
    }));
    m.def("quantize_segments", torch::wrap_pybind_function([](const Tensor& x, const std::shared_ptr<Recipe>& recipe, const Tensor& offsets,
                                                              const Tensor& padded_offsets, int64_t count, int64_t padded, bool rowwise) {
        return segments(x, *recipe, offsets, padded_offsets, count, padded, rowwise);
    }));
    // Each binding is wrapped so that what torch throws (out of memory, an error raised inside a hook) reaches Python as its own type.
    // None: a call for the general path
    m.def("linear", torch::wrap_pybind_function([](const Tensor& x, const py::tuple& layer) -> std::optional<Tensor> {
        Layer l = layer_from(layer);
        if (transformed() || !plain(x) || !takes(l, x.device())) return std::nullopt;
        py::gil_scoped_release release;
        return linear(x, l);
    }));
    m.def("mlp", torch::wrap_pybind_function([](const Tensor& x, const py::tuple& up, const py::tuple& down, int activation) -> std::optional<Tensor> {
        Layer u = layer_from(up), d = layer_from(down);
        if (transformed() || !plain(x) || !takes(u, x.device()) || !takes(d, x.device()) || !pair(*u.recipe, *d.recipe)) return std::nullopt;
        py::gil_scoped_release release;
        return mlp(x, u, d, activation);
    }));
    m.def("experts", torch::wrap_pybind_function([](const Tensor& x, const Tensor& weight, const Tensor& scale, const std::vector<int64_t>& counts,
                                                    const std::shared_ptr<Recipe>& recipe, const py::object& weight_grad) {
        TORCH_CHECK_NOT_IMPLEMENTED(plain(x) && plain(weight) && plain(scale) && !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode),
                                    "the grouped linear has neither forward-mode derivatives nor rules for functorch transforms");
        const at::ScalarType grad = torch::python::detail::py_object_to_dtype(weight_grad);
        py::gil_scoped_release release;
        return experts(x, weight, scale, counts, recipe, grad);
    }));
}

// Native host path of the optimizer and the wire codec: FP8Muon's step over all parameters (buckets of equal-shaped matrices:
// momentum, Newton-Schulz chain, weight update; AdamW for vectors) and FP8Communication's round trip.
//
// Why it is native: the step of one 1024 x 1024 matrix is 20 kernels of 3-9 us (about 170 us) and took 300 us of Python to
// enqueue; per parameter a step costs about 1 us here, and the matrices of a step share their launches where they can.
#include "host.hpp"

#include <c10/core/Event.h>
#include <c10/core/StreamGuard.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <tuple>

using namespace viola_host;

namespace {

// ---------------------------------------------------------------------------------------------------- Newton-Schulz
constexpr float A_COEFFICIENT = 3.4445f;

// The products that orthogonalize [..., rows, cols] in `steps` steps, one after the other; each reads and writes the arena, the last one
// the result.
struct Chain {
    Tensor matrix, result;                                       // (none where the last product goes into the weights)
    Arena arena;
    int dtype = 0;
    float* sums = nullptr;                                       // of squares, where the chain has room for its own
    viola_ns_matrices start{};                                   // the scaled matrix, in front of the products
    std::vector<viola_ns_product> products;
};

// own_sums: with room for its sums of squares. stored: with room for the result; else its last product has nowhere to go yet.
Chain chain_of(const Tensor& matrix_, int64_t steps, bool gram, bool own_sums = true, bool stored = true) {
    TORCH_CHECK(matrix_.is_cuda(), "viola_amd kernels run on the GPU only");
    TORCH_CHECK(matrix_.dim() >= 2 && steps >= 0, "Newton-Schulz takes matrices and a number of steps, got ", matrix_.dim(), " dimensions and ", steps, " steps");
    Chain c;
    c.matrix = matrix_.contiguous();
    const int64_t rows = c.matrix.size(-2), cols = c.matrix.size(-1), m = std::min(rows, cols), n = std::max(rows, cols);
    const int64_t batch = rows * cols ? c.matrix.numel() / (rows * cols) : 0;
    const bool tall = rows > cols;
    const at::ScalarType type = gram ? at::kHalf : at::kBFloat16;
    c.dtype = code_of(type);
    if (stored || steps == 0) c.result = at::empty(c.matrix.sizes(), c.matrix.options().dtype(type));
    if (c.matrix.numel() == 0) return c;
    const bool quintic = !gram || m == n;                        // the plain iteration; else the recurrence on the Gram matrix
    const int64_t wide = 2 * batch * m * n, square = 2 * batch * m * m;
    int64_t x_at[2], s_at[6];
    const int64_t sums_at = own_sums ? c.arena.take(batch * 256 * 4) : -1;
    const int squares = quintic ? 2 : 6;
    for (int64_t& at : x_at) at = c.arena.take(wide);
    for (int i = 0; i < squares; ++i) s_at[i] = c.arena.take(square);
    c.arena.make(c.matrix.device());
    if (own_sums) c.sums = c.arena.as<float>(sums_at);
    void *const into = c.result.defined() ? c.result.mutable_data_ptr() : nullptr;
    void *x = steps ? c.arena.at(x_at[0]) : into, *spare = c.arena.at(x_at[1]);   // no steps: the scaled matrix
    c.start = {c.matrix.const_data_ptr(), x, batch, rows, cols};
    if (steps == 0) return c;
    auto gemm = [&](const void* a, const void* b, bool transpose_b, const void* residual, int epilogue, int64_t out_cols, int64_t k, void* out,
                    float add_diag, void* out_diag, bool transpose_out) {
        c.products.push_back({a, b, residual, out, out_diag, batch, m, out_cols, k, add_diag, transpose_b, epilogue, transpose_out, nullptr, 0, 0});
    };
    if (quintic) {
        void *r = c.arena.at(s_at[0]), *z = c.arena.at(s_at[1]);
        for (int64_t step = 0; step < steps; ++step) {
            const bool last = step == steps - 1;
            void* out = last ? into : spare;
            gemm(x, x, true, nullptr, 0, m, n, r, 0, nullptr, false);
            gemm(r, r, true, r, 1, m, m, z, 0, nullptr, false);  // r = x x^T is symmetric bit for bit: r r = r r^T
            gemm(z, x, false, x, 2, n, m, out, 0, nullptr, tall && last);
            spare = x;
            x = out;
        }
        return c;
    }
    void *r = c.arena.at(s_at[0]), *z = c.arena.at(s_at[1]), *q = c.arena.at(s_at[2]), *q_next = c.arena.at(s_at[3]), *rz = c.arena.at(s_at[4]),
         *r_next = c.arena.at(s_at[5]);
    std::vector<int64_t> segments;
    for (const int64_t length : {std::min<int64_t>(steps, 2), std::max<int64_t>(steps - 2, 0)})
        if (length) segments.push_back(length);
    for (size_t index = 0; index < segments.size(); ++index) {
        const bool last = index + 1 == segments.size();
        gemm(x, x, true, nullptr, 0, m, n, r, 0, nullptr, false);
        for (int64_t i = 0; i < segments[index]; ++i) {
            if (i == 0) {                                        // z and q = z + 3.4445 I from the one product
                gemm(r, r, true, r, 1, m, m, z, A_COEFFICIENT, q, false);
            } else {                                             // r = 3.4445 rz + z rz is symmetric only up to rounding: r r as written
                gemm(r, r, false, r, 1, m, m, z, 0, nullptr, false);
                gemm(z, q, false, q, 2, m, m, q_next, 0, nullptr, false);
                std::swap(q, q_next);
            }
            if (i + 1 < segments[index]) {
                gemm(z, r, false, r, 2, m, m, rz, 0, nullptr, false);
                gemm(z, rz, false, rz, 2, m, m, r_next, 0, nullptr, false);
                std::swap(r, r_next);
            }
        }
        void* out = last ? into : spare;
        gemm(q, x, false, nullptr, 0, n, m, out, 0, nullptr, tall && last);
        spare = x;
        x = out;
    }
    return c;
}

// A last product that could not go into the weights is stored after all.
void store_result(Chain& c) {
    c.result = at::empty(c.matrix.sizes(), c.matrix.options().dtype(c.dtype == VIOLA_F16 ? at::kHalf : at::kBFloat16));
    c.products.back().out = c.result.mutable_data_ptr();
    c.products.back().weights = nullptr;
}

void prepare(const Chain& c, float* sums, viola_stream_t stream) {
    VIOLA_CALL(viola_ns_prepare, c.start.in, code_of(c.matrix.scalar_type()), c.start.out, c.dtype, c.start.batch, c.start.rows, c.start.cols, sums, stream);
}

void multiply(const viola_ns_product& p, int dtype, viola_stream_t stream) {
    VIOLA_CALL(viola_ns_gemm, p.a, p.b, p.residual, p.out, dtype, p.transpose_b, p.epilogue, p.batch, p.m, p.n, p.k, p.add_diag, p.out_diag, p.transpose_out, stream);
}

Arena sums_of(int64_t matrices, const at::Device& device) {
    Arena sums;
    sums.take(matrices * 256 * 4);
    sums.make(device);
    return sums;
}

Tensor newton_schulz(const Tensor& matrix, int64_t steps, bool gram) {
    const Chain c = chain_of(matrix, steps, gram);
    if (c.matrix.numel() == 0) return c.result;
    const viola_stream_t stream = stream_of(c.matrix);
    prepare(c, c.sums, stream);
    for (const viola_ns_product& p : c.products) multiply(p, c.dtype, stream);
    return c.result;
}

// Chains of one type that the tiled kernel takes, at most eight, step by step together: the products of a step are one launch. `sums` holds the
// matrices' sums of squares already, or (have_sums 0) has room for them.
void run_together(const std::vector<Chain>& chains, const Arena& sums, int have_sums, viola_stream_t stream) {
    const int dtype = chains[0].dtype;
    std::vector<viola_ns_matrices> starts;
    size_t steps = 0;
    for (const Chain& c : chains) {
        starts.push_back(c.start);
        steps = std::max(steps, c.products.size());
    }
    int status = VIOLA_TRY(viola_ns_prepare_many, starts.data(), (int)starts.size(), dtype, sums.as<float>(0), have_sums, stream);
    if (status == VIOLA_EUNSUPPORTED) {
        for (const Chain& c : chains) prepare(c, sums.as<float>(0), stream);      // (one after the other: each may overwrite the sums)
    } else check("viola_ns_prepare_many", status);
    std::vector<viola_ns_product> step;
    for (size_t i = 0; i < steps; ++i) {
        step.clear();
        bool into_weights = false;
        for (const Chain& c : chains)
            if (i < c.products.size()) {
                step.push_back(c.products[i]);
                into_weights = into_weights || step.back().weights;
            }
        if (step.size() > 1 || into_weights) VIOLA_CALL(viola_ns_gemm_many, step.data(), (int)step.size(), dtype, stream);
        else multiply(step[0], dtype, stream);
    }
}

// ---------------------------------------------------------------------------------------------------- pointer tables
bool aligned(const void* p, int64_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; }

// Device-side pointer tables, kept while their rows stay the same. Keyed by the stream that fills and reads them.
class Tables {
public:
    const int64_t* get(int kind, const std::vector<int64_t>& shape, int64_t count, int64_t ordinal, std::vector<int64_t>&& rows, const at::Device& device,
                       viola_stream_t stream) {
        Table& t = tables_[std::make_tuple(stream, kind, shape, count, ordinal)];
        if (t.rows != rows) {
            t.rows = std::move(rows);
            t.arena = Arena();                                   // launches in flight may still read the old one: a new place
            t.at = t.arena.take((int64_t)t.rows.size() * 8);
            t.arena.make(device);
            VIOLA_CALL(viola_store_words, t.arena.as<int64_t>(t.at), t.rows.data(), (int64_t)t.rows.size(), stream);
        }
        return t.arena.as<int64_t>(t.at);
    }

private:
    struct Table {
        std::vector<int64_t> rows;
        Arena arena;
        int64_t at = 0;
    };
    std::map<std::tuple<viola_stream_t, int, std::vector<int64_t>, int64_t, int64_t>, Table> tables_;
};
enum { MOMENTUM_TABLE = 0, WEIGHT_TABLE = 1, ADAM_TABLE = 2, ADDRESS_TABLE = 3 };

// One launch for a list of tensors over a table of their pointers. False, with nothing done: they do not fit the table kernel, and
// each takes a launch of its own.
struct MomentumRow {
    Tensor grad, q, scale;
    void* out;                                                   // bf16
    int64_t key, count;
};
bool momentum_together(Tables& tables, const std::vector<int64_t>& shape, int64_t ordinal, const std::vector<MomentumRow>& rows, int64_t tile,
                       float beta, float inv_loss_scale, bool nesterov, int rounding, int64_t step, viola_stream_t stream, float* sums = nullptr, int working = VIOLA_BF16) {
    if (rows.empty() || rows.size() > 65535 || tile < 256) return false;
    const at::ScalarType kind = rows[0].grad.scalar_type();
    std::vector<int64_t> words;
    int64_t tiles = 0;
    for (const MomentumRow& r : rows) {
        if (r.count % tile != 0) return false;
        tiles = std::max(tiles, r.count / tile);
        const void *g = r.grad.const_data_ptr(), *q = r.q.const_data_ptr();
        if (r.grad.scalar_type() != kind || r.grad.numel() != r.count || !r.grad.is_contiguous() || !aligned(g, 4 * r.grad.element_size()) || !aligned(q, 4) ||
            !aligned(r.out, 8))
            return false;
        const int64_t s = (int64_t)r.scale.const_data_ptr(), row[8] = {(int64_t)g, (int64_t)q, s, (int64_t)q, s, (int64_t)r.out, r.key, r.count / tile};
        words.insert(words.end(), row, row + 8);
    }
    const int64_t* t = tables.get(MOMENTUM_TABLE, shape, (int64_t)rows.size(), ordinal, std::move(words), rows[0].q.device(), stream);
    if (sums) VIOLA_CALL(viola_momentum_update_squares, t, (int64_t)rows.size(), tiles, code_of(kind), (int)tile, beta, inv_loss_scale, nesterov, rounding, step, working, sums, stream);
    else VIOLA_CALL(viola_momentum_update_table, t, (int64_t)rows.size(), tiles, code_of(kind), (int)tile, beta, inv_loss_scale, nesterov, rounding, step, stream);
    return true;
}

struct WeightRow {
    Tensor weight;
    const void* update;
};
bool weights_together(Tables& tables, const std::vector<int64_t>& shape, int64_t ordinal, const std::vector<WeightRow>& rows, int64_t count,
                      at::ScalarType update_type, float lr, float weight_decay, float update_scale, viola_stream_t stream) {
    if (rows.empty() || rows.size() > 65535 || count % 4 != 0) return false;
    const int64_t update_bytes = 4 * (int64_t)at::elementSize(update_type);
    std::vector<int64_t> words;
    for (const WeightRow& r : rows) {
        const void* w = r.weight.const_data_ptr();
        if (r.weight.scalar_type() != at::kFloat || r.weight.numel() != count || !r.weight.is_contiguous() || !aligned(w, 16) || !aligned(r.update, update_bytes))
            return false;
        words.push_back((int64_t)w);
        words.push_back((int64_t)r.update);
    }
    const int64_t* t = tables.get(WEIGHT_TABLE, shape, (int64_t)rows.size(), ordinal, std::move(words), rows[0].weight.device(), stream);
    VIOLA_CALL(viola_weight_update_table, t, (int64_t)rows.size(), count, code_of(update_type), lr, weight_decay, update_scale, stream);
    return true;
}

struct AdamRow {
    Tensor weight, grad, first, second;
    int64_t key, offset;
};
struct AdamSettings {
    float lr, weight_decay, b1, b2, inv_c1, inv_c2, eps;
    int rounding;
    int64_t step;                                                // before this one
    bool adamw, maximize;
};
bool adam_together(Tables& tables, const std::vector<AdamRow>& rows, const AdamSettings& a, viola_stream_t stream) {
    if (rows.empty() || rows.size() > 65535) return false;
    const AdamRow& head = rows[0];
    std::vector<int64_t> words;
    int64_t most = 0;
    for (const AdamRow& r : rows) {
        for (const Tensor* t : {&r.weight, &r.grad, &r.first, &r.second})
            if (!t->is_contiguous() || t->numel() != r.weight.numel()) return false;
        if (r.weight.scalar_type() != head.weight.scalar_type() || r.grad.scalar_type() != head.grad.scalar_type() ||
            r.first.scalar_type() != head.first.scalar_type() || r.second.scalar_type() != head.first.scalar_type())
            return false;
        const int64_t row[7] = {(int64_t)r.weight.const_data_ptr(), (int64_t)r.grad.const_data_ptr(), (int64_t)r.first.const_data_ptr(),
                                (int64_t)r.second.const_data_ptr(), r.weight.numel(), r.key, r.offset};
        words.insert(words.end(), row, row + 7);
        most = std::max(most, r.weight.numel());
    }
    // one table per list of equal settings, told apart by what the first row points at
    const int64_t* t = tables.get(ADAM_TABLE, {words[0]}, (int64_t)rows.size(), 0, std::move(words), head.weight.device(), stream);
    VIOLA_CALL(viola_adam_update_table, t, (int64_t)rows.size(), most, code_of(head.weight.scalar_type()), code_of(head.grad.scalar_type()),
               code_of(head.first.scalar_type()), a.lr, a.weight_decay, a.b1, a.b2, a.inv_c1, a.inv_c2, a.eps, a.rounding, a.step, a.adamw, a.maximize, stream);
    return true;
}

// ---------------------------------------------------------------------------------------------------- FP8Muon.step
// One parameter group's settings, read once per step.
struct Group {
    double lr, weight_decay, momentum, b1, b2, eps;
    bool nesterov, batched, gram, match_rms;
    int use_muon;                                                // -1: by the parameter's dimensions
    int granularity, rounding, master_rounding;
    int64_t tile, block_rows, block_cols, seed, master_seed, ns_steps;
    at::ScalarType adam_state;
};

struct Item {
    Tensor param, grad;
    py::dict state;
    const Group* group;
    int64_t index, step;
    Tensor q, scale;                                             // matrices: FP8 momentum and its scales
    Tensor first, second;                                        // vectors: the moments
};

constexpr uint64_t MASK63 = (1ull << 63) - 1;
int64_t rounding_key(int64_t seed, int64_t index, uint64_t stride) { return (int64_t)(((uint64_t)seed + (uint64_t)index * stride) & MASK63); }
int64_t momentum_key(const Item& it) { return rounding_key(it.group->seed, it.index, 0x9E3779B97F4A7C15ull); }
int64_t master_key(const Item& it) { return rounding_key(it.group->master_seed, it.index, 0x517CC1B727220A95ull); }
int rounding_code(const py::handle& h) { return h.cast<std::string>() == "stochastic" ? VIOLA_STOCHASTIC : VIOLA_NEAREST; }

Group read_group(const py::dict& d) {
    Group g;
    auto number = [&](const char* name) { return py::float_(py::object(d[name])).cast<double>(); };
    auto integer = [&](const char* name) { return d[name].cast<int64_t>(); };
    g.lr = number("lr"); g.weight_decay = number("weight_decay"); g.momentum = number("momentum"); g.eps = number("eps");
    const auto betas = py::sequence(py::object(d["betas"])), block = py::sequence(py::object(d["block_shape"]));
    g.b1 = betas[0].cast<double>(); g.b2 = betas[1].cast<double>();
    g.block_rows = block[0].cast<int64_t>(); g.block_cols = block[1].cast<int64_t>();
    g.nesterov = py::bool_(py::object(d["nesterov"])); g.batched = py::bool_(py::object(d["batched"]));
    g.gram = d["ns_method"].cast<std::string>() == "gram";
    g.match_rms = d["adjust_lr_fn"].cast<std::string>() == "match_rms_adamw";
    g.use_muon = d["use_muon"].is_none() ? -1 : (int)(bool)py::bool_(py::object(d["use_muon"]));
    g.granularity = d["granularity"].cast<std::string>() == "tile" ? 0 : 1;
    g.rounding = rounding_code(d["rounding"]);
    g.master_rounding = rounding_code(d["master_rounding"]);
    g.tile = integer("tile_size"); g.seed = integer("rounding_seed"); g.master_seed = integer("master_rounding_seed"); g.ns_steps = integer("ns_steps");
    g.adam_state = torch::python::detail::py_object_to_dtype(d["adam_state_dtype"]);
    return g;
}

// The matrix a parameter stands for: conv filters flatten to [out, -1], batched groups keep their leading dimensions.
std::vector<int64_t> matrix_shape(const Tensor& p, const Group& g) {
    if (g.batched) return p.sizes().vec();
    return {p.size(0), p.size(0) ? p.numel() / p.size(0) : 0};
}

class MuonHost {
public:
    void step(const py::list& work, const py::list& group_list) {
        std::vector<Group> groups;
        std::vector<PyObject*> handles;
        groups.reserve(group_list.size());
        for (const auto& g : group_list) {
            groups.push_back(read_group(g.cast<py::dict>()));
            handles.push_back(g.ptr());
        }
        // buckets in the order their first matrix comes; a bucket that would exceed batch_elements is closed and a new one begins
        std::vector<std::vector<Item>> ready, vectors;
        std::map<std::tuple<std::vector<int64_t>, int, bool, int64_t>, size_t> open;
        using VectorKey = std::tuple<int, int, int, int, double, double, double, double, double, int64_t, int>;
        std::map<VectorKey, size_t> vector_of;
        for (const auto& entry : work) {
            const auto t = entry.cast<py::tuple>();
            Item it{t[0].cast<Tensor>(), t[1].cast<Tensor>(), t[2].cast<py::dict>(), nullptr, t[4].cast<int64_t>(), 0};
            for (size_t i = 0; i < handles.size(); ++i)
                if (handles[i] == t[3].ptr()) it.group = &groups[i];
            TORCH_INTERNAL_ASSERT(it.group);
            TORCH_CHECK(it.param.is_cuda() && !it.grad.is_sparse(), "viola_amd kernels run on the GPU only, on dense gradients");
            const at::ScalarType kind = it.param.scalar_type();
            if (kind != at::kFloat && kind != at::kBFloat16 && kind != at::kHalf) {
                PyErr_SetString(PyExc_AssertionError, "Bind FP8 modules with viola.optim.bind_optimizer before stepping.");
                throw py::error_already_set();
            }
            if (!it.state.contains("step")) it.state["step"] = 0;
            it.step = it.state["step"].cast<int64_t>();
            const Group& g = *it.group;
            const int device = it.param.device().index();
            const bool matrix = g.use_muon < 0 ? it.param.dim() >= 2 : g.use_muon != 0;
            if (!matrix) {
                const VectorKey key{device, (int)kind, (int)it.grad.scalar_type(), (int)g.adam_state, g.lr, g.weight_decay, g.b1, g.b2, g.eps, it.step, g.master_rounding};
                const auto [at, fresh] = vector_of.try_emplace(key, vectors.size());
                if (fresh) vectors.emplace_back();
                prepare_vector(it);
                vectors[at->second].push_back(std::move(it));
                continue;
            }
            prepare_matrix(it);
            const int64_t count = it.param.numel();
            const auto key = std::make_tuple(matrix_shape(it.param, g), device, g.gram, g.ns_steps);
            const auto [at, fresh] = open.try_emplace(key, ready.size());
            if (fresh) ready.emplace_back();
            std::vector<Item>& bucket = ready[at->second];
            bucket.push_back(std::move(it));
            if (((int64_t)bucket.size() + 1) * count > batch_elements) open.erase(at);
        }
        {
            py::gil_scoped_release release;
            step_buckets(ready);
            for (auto& bucket : vectors) step_vectors(bucket);
        }
        for (auto* lists : {&ready, &vectors})
            for (auto& bucket : *lists)
                for (Item& it : bucket) it.state["step"] = it.step + 1;
    }

    int64_t lanes = 4;
    // Equal-shaped matrices of one step go through Newton-Schulz as ONE batched chain (of at most this many elements): every
    // matrix of the batch sees exactly the arithmetic it would see alone, and the launches fill the GPU.
    int64_t batch_elements = 1ll << 28;

    int64_t streams(int device) const {
        const auto at = lanes_.find(device);
        return at == lanes_.end() ? 0 : (int64_t)at->second.size();
    }

private:
    Tables tables_;
    std::map<int, std::vector<c10::Stream>> lanes_;

    // The state is the caller's: it may have been loaded, moved to the host or replaced, and the kernels read it by raw pointer.
    static void check_state(const Item& it, const Tensor& state, int64_t elements, int64_t bytes_each) {
        TORCH_CHECK(state.device() == it.param.device() && state.is_contiguous() && state.numel() >= elements && state.element_size() == bytes_each,
                    "FP8Muon: the state of a parameter of ", it.param.numel(), " elements must be contiguous on ", it.param.device(), " with at least ", elements,
                    " elements of ", bytes_each, " bytes, it has ", state.numel(), " of ", state.element_size(), " on ", state.device());
    }

    // Whatever is refused is refused here, before the first launch: a step that raises has changed nothing.
    static void prepare_vector(Item& it) {
        if (!it.state.contains("exp_avg")) {
            const auto options = at::TensorOptions().dtype(it.group->adam_state);
            it.state["exp_avg"] = py::cast(at::zeros_like(it.param, options));
            it.state["exp_avg_sq"] = py::cast(at::zeros_like(it.param, options));
        }
        it.first = it.state["exp_avg"].cast<Tensor>();
        it.second = it.state["exp_avg_sq"].cast<Tensor>();
        check_state(it, it.first, it.param.numel(), it.first.element_size());
        check_state(it, it.second, it.param.numel(), it.first.element_size());
        TORCH_CHECK(it.param.is_contiguous() && it.first.scalar_type() == it.second.scalar_type() && it.grad.numel() == it.param.numel(),
                    "FP8Muon updates contiguous parameters, with both moments in one type");
    }

    static void prepare_matrix(Item& it) {
        TORCH_CHECK(it.param.dim() >= 2, "Muon updates matrices: a vector in a use_muon=True group");
        TORCH_CHECK(it.param.is_contiguous(), "FP8Muon updates contiguous parameters");
        // 1-D tiles pad the payload to whole tiles, 2-D blocks do not
        const Group& g = *it.group;
        const std::vector<int64_t> shape = matrix_shape(it.param, g);
        const int64_t n = it.param.numel(), rows = shape[shape.size() - 2], cols = shape.back();
        int64_t payload = n, scales = ceil_div(n, g.tile);
        if (g.granularity == 0) payload = scales * g.tile;
        else scales = rows * cols ? n / (rows * cols) * ceil_div(rows, g.block_rows) * ceil_div(cols, g.block_cols) : 0;
        if (!it.state.contains("momentum_q")) {
            const auto options = at::TensorOptions().device(it.param.device());
            it.state["momentum_q"] = py::cast(at::zeros({payload}, options.dtype(at::kByte)));
            it.state["momentum_scale"] = py::cast(at::ones({scales}, options.dtype(at::kFloat)));
        }
        it.q = it.state["momentum_q"].cast<Tensor>();
        it.scale = it.state["momentum_scale"].cast<Tensor>();
        check_state(it, it.q, payload, 1);
        check_state(it, it.scale, scales, 4);
    }

    // The chains of different buckets are independent, and a single chain leaves the GPU partly idle at every launch boundary
    // (a Newton-Schulz GEMM of 28 matrices is ~590 tiles for 512 tile slots: its second round is nearly empty). Buckets
    // that step_together does not take go to up to `lanes` streams of default priority, so the blocks of one chain fill the tails of the
    // others; the caller's stream waits for all of them at the end.
    void step_buckets(std::vector<std::vector<Item>>& ready) {
        // buckets of one shape and size (a shape split because it exceeds batch_elements) each keep their own pointer tables
        std::map<std::pair<std::vector<int64_t>, size_t>, int64_t> seen;
        std::vector<int64_t> ordinals;
        bool one_device = true;
        for (const auto& bucket : ready) {
            ordinals.push_back(seen[{matrix_shape(bucket[0].param, *bucket[0].group), bucket.size()}]++);
            one_device = one_device && bucket[0].param.device() == ready[0][0].param.device();
        }
        if (one_device && step_together(ready)) return;
        if (ready.size() < 2 || lanes < 2 || !one_device) {
            for (size_t i = 0; i < ready.size(); ++i) step_bucket(ready[i], ordinals[i]);
            return;
        }
        const at::Device device = ready[0][0].param.device();
        const c10::impl::VirtualGuardImpl guard(device.type());
        std::vector<c10::Stream>& streams = lanes_[device.index()];
        const size_t used = std::min<size_t>(lanes, ready.size());
        while (streams.size() < used) streams.push_back(guard.getStreamFromGlobalPool(device, false));
        const c10::Stream main = guard.getStream(device);
        c10::Event start(device.type());
        start.record(main);
        // the caller's stream waits for the lanes however this ends (an allocation may fail on the way): what they read is freed there
        struct Join {
            std::vector<c10::Stream>& streams;
            size_t used;
            c10::Stream main;
            bool done = false;
            void now() {
                done = true;
                for (size_t i = 0; i < used; ++i) {
                    c10::Event event(main.device_type());
                    event.record(streams[i]);
                    event.block(main);
                }
            }
            ~Join() {
                try {
                    if (!done) now();
                } catch (...) {                                  // already on the way out with an error
                }
            }
        } join{streams, used, main};
        // largest chains first, one lane after the other: the long ones start together and the short ones pack behind
        std::vector<size_t> order(ready.size());
        for (size_t i = 0; i < order.size(); ++i) order[i] = i;
        auto elements = [&](size_t i) { return (int64_t)ready[i].size() * ready[i][0].param.numel(); };
        std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return elements(a) > elements(b); });
        for (size_t slot = 0; slot < order.size(); ++slot) {
            const c10::Stream lane = streams[slot % used];
            if (slot < used) start.block(lane);
            const c10::StreamGuard on(lane);
            step_bucket(ready[order[slot]], ordinals[order[slot]]);
        }
        join.now();
    }

    // The chains of all buckets step by step together, a product of each in one launch, and one launch each for the momentum with the sums
    // of squares and for the scaling in front of the chains: 17 launches where buckets on lanes of their own took about 80 and the events that
    // join them, which is all that a step of small matrices costs (one block of width 192: 253 -> 99 us, four of 256 316 -> 140, eight of
    // 384 362 -> 325). Large sets gain by the mix of tile lengths (by that alone 28 blocks of width 1152 12560 -> 12280 us, eight of 1280 5842 ->
    // 5185). The recurrence on the Gram matrix gains less there: its launches are several rounds of short tiles with a tail each, which lanes
    // fill, so beyond TOGETHER_GRAM it keeps the lanes. On lanes and together, us, by the sum of m m (m + n): 28 blocks of 256 (7.5e9) 571, 400; two of 640
    // (8.4e9) 386, 314; four of 512 (8.6e9) 400, 316; 23 of 288 (8.8e9) 532, 515; 20 of 320 (1.05e10) 517, 524; four of 640 (1.7e10) 480, 471; ten of 512
    // (2.1e10) 593, 589; 28 of 384 (2.5e10) 803, 835; two of 1024 (3.4e10) 719, 653; 19 of 608 (6.8e10) 1666, 1706.
    static constexpr double TOGETHER_GRAM = 1e10;                // sum of m m (m + n) over the matrices
    // All arenas are held at once, 10 bytes per element at most (5.4 GB); and no more elements than the buckets on lanes may hold.
    static constexpr int64_t TOGETHER_ELEMENTS = 1ll << 29;
    bool step_together(std::vector<std::vector<Item>>& ready) {
        if (ready.empty() || ready.size() > 8) return false;
        const Item& head = ready[0][0];
        const Group& g = *head.group;
        const viola_stream_t stream = stream_of(head.param);
        // what momentum_together would refuse, before anything is allocated or copied for it; and a chain of no product leaves none for the weights
        if (g.tile < 256 || g.ns_steps < 1) return false;
        int64_t elements = 0, parameters = 0;
        double work = 0;
        for (const auto& bucket : ready)
            for (const Item& it : bucket) {
                const Group& h = *it.group;
                const std::vector<int64_t> shape = matrix_shape(it.param, h);
                if (it.param.numel() == 0 || it.param.numel() % h.tile || h.granularity != 0 || it.step != head.step || h.tile != g.tile || h.momentum != g.momentum ||
                    h.nesterov != g.nesterov || h.rounding != g.rounding || h.gram != g.gram || h.ns_steps != g.ns_steps || h.lr != g.lr ||
                    h.weight_decay != g.weight_decay || h.match_rms != g.match_rms || shape.back() % 8 || shape[shape.size() - 2] % 8)
                    return false;
                if (it.param.scalar_type() != at::kFloat || !aligned(it.param.const_data_ptr(), 16)) return false;
                if (it.grad.scalar_type() != head.grad.scalar_type() || it.grad.numel() != it.param.numel() || !aligned(it.q.const_data_ptr(), 4) ||
                    (it.grad.is_contiguous() && !aligned(it.grad.const_data_ptr(), 4 * it.grad.element_size())) || ++parameters > 65535)
                    return false;
                elements += it.param.numel();
                work += (double)it.param.numel() * (double)std::min(shape.back(), shape[shape.size() - 2]) *
                        (1. + (double)std::min(shape.back(), shape[shape.size() - 2]) / (double)std::max(shape.back(), shape[shape.size() - 2]));
            }
        if (elements > TOGETHER_ELEMENTS || elements / std::max<int64_t>(lanes, 1) > batch_elements || (g.gram && work > TOGETHER_GRAM)) return false;
        std::vector<MomentumRow> momentum_rows;
        std::vector<Tensor> inputs;
        for (const auto& bucket : ready) {
            const std::vector<int64_t> shape = matrix_shape(bucket[0].param, *bucket[0].group);
            const int64_t count = bucket[0].param.numel(), rows = shape[shape.size() - 2], cols = shape.back();
            inputs.push_back(at::empty({(int64_t)bucket.size(), count / (rows * cols), rows, cols}, at::TensorOptions().dtype(at::kBFloat16).device(head.param.device())));
            char* out = static_cast<char*>(inputs.back().mutable_data_ptr());
            for (const Item& it : bucket) {
                momentum_rows.push_back({it.grad.contiguous(), it.q, it.scale, out, momentum_key(it), count});
                out += 2 * count;
            }
        }
        // a parameter that is one matrix (not a batch of them): its sum of squares comes with its momentum
        int64_t matrices = 0;
        for (const Tensor& input : inputs) matrices += input.size(0) * input.size(1);
        const bool single = matrices == (int64_t)momentum_rows.size();
        const Arena sums = sums_of(matrices, head.param.device());
        TORCH_INTERNAL_ASSERT(momentum_together(tables_, {}, (int64_t)g.gram, momentum_rows, g.tile, (float)g.momentum, 1.0f, g.nesterov, g.rounding, head.step,
                                                stream, single ? sums.as<float>(0) : nullptr, g.gram ? VIOLA_F16 : VIOLA_BF16));
        std::vector<Chain> chains;
        for (const Tensor& input : inputs) chains.push_back(chain_of(input, g.ns_steps, g.gram, false, false));
        // the last products of the chains go into the weights
        std::vector<int64_t> addresses;
        for (size_t i = 0; i < ready.size(); ++i)
            for (const Item& it : ready[i])
                for (int64_t plane = 0; plane < chains[i].matrix.size(1); ++plane)
                    addresses.push_back((int64_t)it.param.const_data_ptr() + plane * chains[i].matrix.size(-2) * chains[i].matrix.size(-1) * 4);
        const int64_t* at = tables_.get(ADDRESS_TABLE, {}, (int64_t)addresses.size(), (int64_t)g.gram, std::move(addresses), head.param.device(), stream);
        for (Chain& c : chains) {
            into_weights(c.products.back(), at, g, c.matrix.size(-2), c.matrix.size(-1));
            at += c.start.batch;
        }
        run_together(chains, sums, single, stream);
        return true;
    }

    static double update_scale(const Group& g, int64_t rows, int64_t cols) {
        return g.match_rms ? .2 * std::pow((double)std::max(rows, cols), .5) : std::pow(std::max(1., (double)rows / (double)cols), .5);
    }

    // weight = weight * (1 - lr decay) - lr scale update, with the FP32 roundings of viola_weight_update
    static void into_weights(viola_ns_product& last, const int64_t* weights, const Group& g, int64_t rows, int64_t cols) {
        const float lr = (float)g.lr, decayed = lr * (float)g.weight_decay;
        last.weights = weights;
        last.keep = 1.0f - decayed;
        last.rate = lr * (float)update_scale(g, rows, cols);
    }

    void step_bucket(std::vector<Item>& bucket, int64_t ordinal) {
        const Item& head = bucket[0];
        const Group& g = *head.group;
        const std::vector<int64_t> shape = matrix_shape(head.param, g);
        const int64_t size = (int64_t)bucket.size(), count = head.param.numel(), rows = shape[shape.size() - 2], cols = shape.back();
        if (count == 0) return;
        const at::Device device = head.param.device();
        const viola_stream_t stream = stream_of(head.param);
        const Tensor updates_in = at::empty({size, count / (rows * cols), rows, cols}, at::TensorOptions().dtype(at::kBFloat16).device(device));
        char* out = static_cast<char*>(updates_in.mutable_data_ptr());
        std::vector<Tensor> grads;
        for (Item& it : bucket) grads.push_back(it.grad.contiguous());

        // ---- momentum: one launch for the bucket when its members share the recipe and fit the table kernel, else one each
        bool together = g.granularity == 0;
        std::vector<MomentumRow> momentum_rows;
        for (size_t i = 0; together && i < bucket.size(); ++i) {
            const Item& it = bucket[i];
            const Group& h = *it.group;
            together = it.step == head.step && h.granularity == g.granularity && h.tile == g.tile && h.momentum == g.momentum && h.nesterov == g.nesterov &&
                       h.rounding == g.rounding;
            momentum_rows.push_back({grads[i], it.q, it.scale, out + 2 * count * i, momentum_key(it), count});
        }
        if (!together || !momentum_together(tables_, shape, ordinal, momentum_rows, g.tile, (float)g.momentum, 1.0f, g.nesterov, g.rounding, head.step, stream)) {
            for (size_t i = 0; i < bucket.size(); ++i) {
                const Item& it = bucket[i];
                const Group& h = *it.group;
                const bool blocks = h.granularity == 1;
                void* q = it.q.mutable_data_ptr();
                float* s = static_cast<float*>(it.scale.mutable_data_ptr());
                VIOLA_CALL(viola_momentum_update, grads[i].const_data_ptr(), code_of(grads[i].scalar_type()), q, s, q, s, out + 2 * count * i, count, (float)h.momentum,
                           1.0f, h.nesterov, h.granularity, blocks ? 0 : (int)h.tile, blocks ? count / (rows * cols) : 1, blocks ? rows : 1, blocks ? cols : 1,
                           blocks ? (int)h.block_rows : 1, blocks ? (int)h.block_cols : 1, h.rounding, it.step, momentum_key(it), stream);
            }
        }

        // ---- the chain, its last product into the weights where they allow it
        together = true;
        bool in_place = rows % 8 == 0 && cols % 8 == 0 && g.ns_steps > 0;
        for (const Item& it : bucket) {
            const Group& h = *it.group;
            together = together && h.lr == g.lr && h.weight_decay == g.weight_decay && h.match_rms == g.match_rms;
            in_place = in_place && it.param.scalar_type() == at::kFloat && aligned(it.param.const_data_ptr(), 16);
        }
        // (of any size: a launch less, and 8 bytes per element. us, with a launch for the weights and without: one block of 192 335, 324; eight of 384 379,
        // 364; two of 768 418, 403; eight of 1024 2453, 2361)
        in_place = in_place && together;
        Chain chain = chain_of(updates_in, g.ns_steps, g.gram, true, !in_place);
        prepare(chain, chain.sums, stream);
        for (size_t i = 0; i + 1 < chain.products.size(); ++i) multiply(chain.products[i], chain.dtype, stream);
        if (in_place) {
            std::vector<int64_t> addresses;
            for (const Item& it : bucket)
                for (int64_t plane = 0; plane < chain.matrix.size(1); ++plane) addresses.push_back((int64_t)it.param.const_data_ptr() + plane * rows * cols * 4);
            viola_ns_product& last = chain.products.back();
            into_weights(last, tables_.get(ADDRESS_TABLE, shape, (int64_t)addresses.size(), ordinal, std::move(addresses), device, stream), g, rows, cols);
            const int status = VIOLA_TRY(viola_ns_gemm_many, &last, 1, chain.dtype, stream);
            if (status == 0) return;
            if (status != VIOLA_EUNSUPPORTED) check("viola_ns_gemm_many", status);
            store_result(chain);                                 // a matrix of 2 GB and more
        }
        if (!chain.products.empty()) multiply(chain.products.back(), chain.dtype, stream);

        // ---- weights
        const Tensor updates = chain.result;
        const char* from = static_cast<const char*>(updates.const_data_ptr());
        const int update_code = code_of(updates.scalar_type());
        std::vector<WeightRow> weight_rows;
        for (size_t i = 0; i < bucket.size(); ++i) weight_rows.push_back({bucket[i].param, from + 2 * count * i});
        if (together && weights_together(tables_, shape, ordinal, weight_rows, count, updates.scalar_type(), (float)g.lr, (float)g.weight_decay,
                                         (float)update_scale(g, rows, cols), stream))
            return;
        for (size_t i = 0; i < bucket.size(); ++i) {
            const Item& it = bucket[i];
            const Group& h = *it.group;
            VIOLA_CALL(viola_weight_update, it.param.mutable_data_ptr(), code_of(it.param.scalar_type()), from + 2 * count * i, update_code, count, (float)h.lr,
                       (float)h.weight_decay, (float)update_scale(h, rows, cols), h.master_rounding, it.step, master_key(it), 0, stream);
        }
    }

    // Vectors (biases, norms, modulation tables) are a few thousand elements each: those that share dtypes, hyper-parameters
    // and step count take AdamW in one launch over a table of their pointers.
    void step_vectors(std::vector<Item>& bucket) {
        const Item& head = bucket[0];
        const Group& g = *head.group;
        const viola_stream_t stream = stream_of(head.param);
        const double step = (double)(head.step + 1);
        const float inv_c1 = (float)(1. / (1. - std::pow(g.b1, step))), inv_c2 = (float)(1. / (1. - std::pow(g.b2, step)));
        const int weight_code = code_of(head.param.scalar_type()), grad_code = code_of(head.grad.scalar_type());
        std::vector<AdamRow> rows;
        std::vector<Tensor> grads;
        for (const Item& it : bucket) {
            rows.push_back({it.param, it.grad, it.first, it.second, master_key(it), 0});
            grads.push_back(it.grad.contiguous());
        }
        const AdamSettings settings{(float)g.lr, (float)g.weight_decay, (float)g.b1, (float)g.b2, inv_c1, inv_c2, (float)g.eps, g.master_rounding, head.step, true, false};
        if (bucket.size() > 1 && adam_together(tables_, rows, settings, stream)) return;
        for (size_t i = 0; i < bucket.size(); ++i) {
            const Item& it = bucket[i];
            if (it.param.numel() == 0) continue;
            VIOLA_CALL(viola_adam_update, it.param.mutable_data_ptr(), weight_code, grads[i].const_data_ptr(), grad_code, it.first.mutable_data_ptr(),
                       it.second.mutable_data_ptr(), code_of(it.first.scalar_type()), it.param.numel(), (float)g.lr, (float)g.weight_decay, (float)g.b1, (float)g.b2,
                       inv_c1, inv_c2, (float)g.eps, g.master_rounding, it.step, master_key(it), 0, 1, 0, stream);
        }
    }
};

// ---------------------------------------------------------------------------------------------------- wire codec
// value <- decode(encode(value)) through the packet buffer
void roundtrip(const Tensor& value, const Tensor& send, int64_t tile, py::object format) {
    const int code = code_of(torch::python::detail::py_object_to_dtype(format));
    TORCH_CHECK(value.is_cuda() && value.scalar_type() == at::kFloat && value.is_contiguous(), "the codec takes contiguous FP32 values on the GPU");
    TORCH_CHECK(send.device() == value.device() && send.scalar_type() == at::kByte && send.is_contiguous(), "the packet buffer is on ", send.device(), ", the values on ", value.device());
    const int64_t groups = ceil_div(value.numel(), tile);
    TORCH_CHECK(ceil_to(groups * (tile + 4), 16) <= send.numel(), "the bucket exceeds the codec's capacity");
    if (value.numel() == 0) return;
    const viola_stream_t stream = stream_of(value);
    float* x = static_cast<float*>(value.mutable_data_ptr());
    void* packet = send.mutable_data_ptr();
    const int status = VIOLA_TRY(viola_comm_roundtrip, x, value.numel(), packet, groups, (int)tile, code, stream);
    if (status == 0) return;
    if (status != VIOLA_EUNSUPPORTED) check("viola_comm_roundtrip", status);
    VIOLA_CALL(viola_comm_pack, x, value.numel(), packet, 1, groups, (int)tile, code, stream);
    VIOLA_CALL(viola_comm_unpack, packet, x, value.numel(), 1, groups, (int)tile, code, 0, stream);
}

}  // namespace

namespace viola_host {

void register_optimizer(py::module_& m) {
    m.def("newton_schulz", torch::wrap_pybind_function_no_gil(newton_schulz), py::arg("matrix"), py::arg("steps"), py::arg("gram"));
    m.def("roundtrip", torch::wrap_pybind_function(roundtrip));
    // The table launches of FP8Muon's step as operators of their own (optim/_kernels.py); the lists are one entry per tensor.
    py::class_<Tables, std::shared_ptr<Tables>>(m, "Tables").def(py::init<>());
    m.def("momentum_update_many", torch::wrap_pybind_function([](Tables& tables, const std::vector<Tensor>& grads, const std::vector<Tensor>& qs,
                                                                 const std::vector<Tensor>& scales, const std::vector<Tensor>& outs, const std::vector<int64_t>& keys,
                                                                 int64_t tile, double beta, double inv_loss_scale, bool nesterov, int rounding, int64_t step) {
        std::vector<MomentumRow> rows;
        for (size_t i = 0; i < grads.size(); ++i) {
            TORCH_CHECK(grads[i].is_cuda() && qs[i].is_cuda() && scales[i].is_cuda() && outs[i].is_cuda(), "viola_amd kernels run on the GPU only");
            if (outs[i].scalar_type() != at::kBFloat16 || outs[i].numel() < grads[i].numel()) return false;
            rows.push_back({grads[i], qs[i], scales[i], outs[i].mutable_data_ptr(), keys[i], grads[0].numel()});
        }
        return momentum_together(tables, {}, 0, rows, tile, (float)beta, (float)inv_loss_scale, nesterov, rounding, step, stream_of(grads[0]));
    }));
    m.def("weight_update_many", torch::wrap_pybind_function([](Tables& tables, const std::vector<Tensor>& weights, const std::vector<Tensor>& updates, double lr,
                                                               double weight_decay, double update_scale) {
        std::vector<WeightRow> rows;
        for (size_t i = 0; i < weights.size(); ++i) {
            TORCH_CHECK(weights[i].is_cuda() && updates[i].is_cuda(), "viola_amd kernels run on the GPU only");
            if (updates[i].scalar_type() != updates[0].scalar_type() || updates[i].numel() != weights[i].numel() || !updates[i].is_contiguous()) return false;
            rows.push_back({weights[i], updates[i].const_data_ptr()});
        }
        return weights_together(tables, {}, 0, rows, weights[0].numel(), updates[0].scalar_type(), (float)lr, (float)weight_decay, (float)update_scale,
                                stream_of(weights[0]));
    }));
    m.def("adam_update_many", torch::wrap_pybind_function([](Tables& tables, const std::vector<Tensor>& weights, const std::vector<Tensor>& grads,
                                                             const std::vector<Tensor>& firsts, const std::vector<Tensor>& seconds, const std::vector<int64_t>& keys,
                                                             const std::vector<int64_t>& offsets, const std::vector<double>& hyper, int rounding, int64_t step,
                                                             bool adamw, bool maximize) {
        std::vector<AdamRow> rows;
        for (size_t i = 0; i < weights.size(); ++i) {
            TORCH_CHECK(weights[i].is_cuda() && grads[i].is_cuda() && firsts[i].is_cuda() && seconds[i].is_cuda(), "viola_amd kernels run on the GPU only");
            rows.push_back({weights[i], grads[i], firsts[i], seconds[i], keys[i], offsets[i]});
        }
        const AdamSettings settings{(float)hyper[0], (float)hyper[1], (float)hyper[2], (float)hyper[3], (float)hyper[4], (float)hyper[5], (float)hyper[6], rounding, step,
                                    adamw, maximize};
        return adam_together(tables, rows, settings, stream_of(weights[0]));
    }));
    py::class_<MuonHost>(m, "MuonHost").def(py::init<>())
        .def("step", torch::wrap_pybind_function([](MuonHost& host, const py::list& work, const py::list& groups) { host.step(work, groups); }))
        .def_readwrite("lanes", &MuonHost::lanes).def_readwrite("batch_elements", &MuonHost::batch_elements).def("streams", &MuonHost::streams);
}

}  // namespace viola_host

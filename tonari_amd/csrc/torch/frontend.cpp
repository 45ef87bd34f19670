// The device search of the PyTorch frontend in native code: one call sizes
// and allocates the workspace and outputs, drives the C ABI
// (include/tonari_hip.h) on torch's current stream and attaches the gradient
// of d and D.  It holds no state: what a repeated call reserves (capacity,
// plan, bins, hit-mask words) comes from and goes back to the caller, as do
// the pinned status words and their event.
//
// Replaces the call into the reference's pybind11 module and its quantity
// assembly (src/tonari/_torch_frontend.py:78-158); the sequence of native
// calls is described in tonari_amd/_torch_frontend.py.
//
// Why native: small calls are bound by the host.  For one 16-atom crystal
// with forces the same steps in Python (ctypes structures, allocations, an
// autograd.Function whose backward takes the GIL in the engine's thread)
// took 252 us per call against 70 us of kernels, and take 126 us here; 256
// crystals with forces 243 -> 160 us, one molecule's list 71 -> 43 us.

#include "../../../include/tonari_hip.h"

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>
#include <torch/version.h>

#include <cstring>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr size_t kErrLen = 512;

void* current_stream(const Tensor& t) {
    return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

int32_t dtype_code(const Tensor& t) {
    return t.scalar_type() == at::kFloat ? TNR_FLOAT32 : TNR_FLOAT64;
}

template <typename T>
T* ptr(const std::optional<Tensor>& t) {
    return t && t->defined() ? (T*)t->data_ptr() : nullptr;
}

// ------------------------------------------------------------- gradients

// D by the reference's Torch expression (_torch_frontend.py:92-101).
Tensor torch_vectors(const Tensor& positions, const Tensor& cell, const Tensor& batch_ptr,
                     const Tensor& pairs, const Tensor& shifts) {
    const Tensor source = pairs.select(1, 0).contiguous();
    const Tensor target = pairs.select(1, 1).contiguous();
    const Tensor batch =
        at::bucketize(source, batch_ptr.slice(0, 1), /*out_int32=*/false, /*right=*/true);
    return positions.index({target}) - positions.index({source}) +
           at::einsum("ei,eij->ej", {shifts.to(positions.scalar_type()), cell.index({batch})});
}

// D (and d) as the emitting kernel wrote them, differentiable in positions
// and cell: the gradient of the reference's expression in one kernel
// (tnr_backward_list).  When a graph of the gradient is asked for
// (create_graph), the same gradient comes from that Torch expression, so
// that higher derivatives exist.  An output without a gradient reaches the
// backward undefined, not as a zero tensor to fill and read.
struct FusedGeometry : torch::autograd::Function<FusedGeometry> {
    static variable_list forward(AutogradContext* ctx, const Tensor& positions, const Tensor& cell,
                                 const Tensor& pairs, const Tensor& shifts, const Tensor& batch_ptr,
                                 const Tensor& vectors, const std::optional<Tensor>& distances,
                                 const std::optional<Tensor>& runs) {
        ctx->save_for_backward({positions, cell, pairs, shifts, batch_ptr, vectors,
                                distances ? *distances : Tensor(), runs ? *runs : Tensor()});
        ctx->set_materialize_grads(false);
        variable_list out{vectors.view_as(vectors)};
        if (distances) out.push_back(distances->view_as(*distances));
        return out;
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &positions = saved[0], &cell = saved[1], &pairs = saved[2], &shifts = saved[3],
                     &batch_ptr = saved[4], &vectors = saved[5], &distances = saved[6],
                     &runs = saved[7];
        const Tensor gv = grads[0];
        const Tensor gd = grads.size() > 1 ? grads[1] : Tensor();
        const bool need_pos = ctx->needs_input_grad(0), need_cell = ctx->needs_input_grad(1);
        variable_list out(8);
        if (!gv.defined() && !gd.defined()) return out;
        if (at::GradMode::is_enabled()) {
            const Tensor D = torch_vectors(positions, cell, batch_ptr, pairs, shifts);
            variable_list outputs, upstream, wrt;
            if (gv.defined()) {
                outputs.push_back(D);
                upstream.push_back(gv);
            }
            if (gd.defined()) {
                outputs.push_back(at::linalg_vector_norm(D, 2, at::IntArrayRef{1}));
                upstream.push_back(gd);
            }
            if (need_pos) wrt.push_back(positions);
            if (need_cell) wrt.push_back(cell);
            const variable_list found = torch::autograd::grad(
                outputs, wrt, upstream, std::nullopt, /*create_graph=*/true, /*allow_unused=*/true);
            size_t k = 0;
            if (need_pos) out[0] = found[k++];
            if (need_cell) out[1] = found[k];
            return out;
        }
        c10::DeviceGuard guard(positions.device());
        const Tensor gvc = gv.defined() ? gv.contiguous() : gv;
        const Tensor gdc = gd.defined() ? gd.contiguous() : gd;
        const Tensor grad_positions = at::empty(positions.sizes(), positions.options());
        const Tensor grad_cell = at::empty(cell.sizes(), cell.options());
        tnr_backward r{};
        r.dtype = dtype_code(positions);
        r.n_pairs = pairs.size(0);
        r.n_atoms = positions.size(0);
        r.n_structures = batch_ptr.numel() - 1;
        r.batch_ptr = (const int64_t*)batch_ptr.data_ptr();
        r.pairs = (const int64_t*)pairs.data_ptr();
        r.shifts = (const int32_t*)shifts.data_ptr();
        r.vectors = vectors.data_ptr();
        r.distances = distances.defined() ? distances.data_ptr() : nullptr;
        r.grad_vectors = gvc.defined() ? gvc.data_ptr() : nullptr;
        r.grad_distances = gdc.defined() ? gdc.data_ptr() : nullptr;
        r.grad_positions = grad_positions.data_ptr();
        r.grad_cell = grad_cell.data_ptr();
        r.source_runs = runs.defined() ? runs.data_ptr() : nullptr;
        char err[kErrLen] = {0};
        void* stream = current_stream(positions);
        int code = tnr_zero_gradients(&r, stream, err, kErrLen);
        if (code == TNR_OK) code = tnr_backward_list(&r, stream, err, kErrLen);
        TORCH_CHECK_VALUE(code != TNR_INPUT_ERROR, err);
        TORCH_CHECK(code == TNR_OK, err);
        if (need_pos) out[0] = grad_positions;
        if (need_cell) out[1] = grad_cell;
        return out;
    }
};

// (D, d or None) carrying the gradient.
std::tuple<Tensor, std::optional<Tensor>> fused_geometry(
    const Tensor& positions, const Tensor& cell, const Tensor& pairs, const Tensor& shifts,
    const Tensor& batch_ptr, const Tensor& vectors, const std::optional<Tensor>& distances,
    const std::optional<Tensor>& runs) {
    const variable_list out = FusedGeometry::apply(positions, cell, pairs, shifts, batch_ptr,
                                                   vectors, distances, runs);
    return {out[0], out.size() > 1 ? std::optional<Tensor>(out[1]) : std::nullopt};
}

// ---------------------------------------------------------------- search

// The rows of the requested quantities, `rows` of each.
struct Rows {
    std::optional<Tensor> P, S, i, j, d, D, E;

    void allocate(const std::string& want, int64_t rows, const Tensor& like) {
        const auto real = like.options();
        const auto i64 = real.dtype(at::kLong), i32 = real.dtype(at::kInt);
        for (const char c : want) switch (c) {
                case 'P': P = at::empty({rows, 2}, i64); break;
                case 'S': S = at::empty({rows, 3}, i32); break;
                case 'i': i = at::empty({rows}, i64); break;
                case 'j': j = at::empty({rows}, i64); break;
                case 'd': d = at::empty({rows}, real); break;
                case 'D': D = at::empty({rows, 3}, real); break;
                default: E = at::empty({2 * rows}, i64); break;  // edge-first index
            }
    }
    tnr_outputs outputs(int64_t rows, int64_t plan, int64_t bins) const {
        tnr_outputs o{};
        o.n_pairs = rows;
        o.plan = plan;
        o.n_tasks = bins;
        o.pairs = ptr<int64_t>(P);
        o.shifts = ptr<int32_t>(S);
        o.distances = ptr<void>(d);
        o.vectors = ptr<void>(D);
        o.sources = ptr<int64_t>(i);
        o.targets = ptr<int64_t>(j);
        o.edge_index = ptr<int64_t>(E);
        return o;
    }
    // The first `count` rows; the edge-first index as (2, count).
    void trim(int64_t count, int64_t rows) {
        if (E) E = E->slice(0, 0, 2 * count).view({2, count});
        if (count == rows) return;
        for (auto* t : {&P, &S, &i, &j, &d, &D})
            if (*t) *t = (*t)->slice(0, 0, count);
    }
    Tensor get(char c) const {
        switch (c) {
            case 'P': return *P;
            case 'S': return *S;
            case 'i': return *i;
            case 'j': return *j;
            case 'd': return *d;
            case 'D': return *D;
            default: return *E;
        }
    }
};

// What a call of the shape reserves (None: the shape's first call).
using Guess = std::tuple<int64_t, int64_t, int64_t, int64_t>;  // rows, plan, bins, mask words

// What became of the writing pass sized by the guess.
enum Reserved : int { kUnused = 0, kFitted = 1, kMissed = 2, kNoMemory = 3 };

// (code, message, tensors in the order of `quantities`, (E, plan, bins, mask
// words wanted), Reserved); with a code other than TNR_OK only the message is
// set.
using Answer = std::tuple<int, std::string, std::vector<Tensor>, Guess, int>;

Answer search(const std::string& quantities, const Tensor& positions, const Tensor& cell,
              const Tensor& pbc, const Tensor& batch_ptr, double cutoff, int64_t algorithm,
              bool sorted, bool half_list, bool include_self, bool need_grad,
              const std::optional<Guess>& guess, int64_t host, int64_t event, int64_t run_pairs,
              int64_t run_atoms) {
    c10::DeviceGuard guard(positions.device());
    const Tensor pos = positions.detach().contiguous(), cel = cell.detach().contiguous();
    const Tensor bp = batch_ptr.contiguous(), flags = pbc.contiguous();
    void* stream = current_stream(pos);
    auto* words = (int64_t*)host;
    std::string want;
    for (const char c : quantities)
        if (want.find(c) == std::string::npos) want += c;
    if (need_grad)
        // what the backward reads (d only where d itself can have a gradient)
        for (const char c : {'P', 'S', 'D'})
            if (want.find(c) == std::string::npos) want += c;

    tnr_request req{};
    req.dtype = dtype_code(pos);
    req.algorithm = (int32_t)algorithm;
    req.n_atoms = pos.size(0);
    req.n_structures = bp.numel() - 1;
    req.positions = pos.data_ptr();
    req.batch_ptr = (const int64_t*)bp.data_ptr();
    req.cell = cel.data_ptr();
    req.pbc = (const uint8_t*)flags.data_ptr();
    req.cutoff = cutoff;
    req.half_list = half_list;
    req.include_self = include_self;
    req.sorted = sorted;
    // hit-mask rows sized by the earlier calls of the shape (first call: the
    // library's default)
    req.mask_words = guess ? (int32_t)std::get<3>(*guess) : 0;
    const size_t ws_bytes = tnr_workspace_size(&req);
    const Tensor workspace = at::empty({(int64_t)ws_bytes}, pos.options().dtype(at::kByte));
    void* ws = workspace.data_ptr();

    char err[kErrLen] = {0};
    const auto failed = [&](int code) { return Answer{code, err, {}, {}, kUnused}; };
    // records the event behind the count and waits for it
    const auto record = [&]() {
        const hipError_t e = hipEventRecord((hipEvent_t)event, (hipStream_t)stream);
        TORCH_CHECK(e == hipSuccess, hipGetErrorString(e));
    };
    const auto wait = [&]() {
        const hipError_t e = hipEventSynchronize((hipEvent_t)event);
        TORCH_CHECK(e == hipSuccess, hipGetErrorString(e));
    };
    // the previous plan is the count's hint (the device checks it)
    int code = tnr_count_async_hinted(&req, ws, ws_bytes, words, stream,
                                      guess ? std::get<1>(*guess) : -1, err, kErrLen);
    if (code != TNR_OK) return failed(code);
    record();
    Rows out;
    int64_t rows = 0;
    int reserved = kUnused;
    if (guess && !want.empty()) {
        rows = std::get<0>(*guess);
        reserved = kMissed;
        try {
            out.allocate(want, rows, pos);
        } catch (const c10::OutOfMemoryError&) {
            // the list itself may still fit, in whole segments: the rows that
            // were allocated would be split for it and keep their rest
            out = Rows{};
            c10::hip::HIPCachingAllocator::emptyCache();
            reserved = kNoMemory;
        }
    }
    if (reserved == kMissed) {
        const tnr_outputs o = out.outputs(rows, std::get<1>(*guess), std::get<2>(*guess));
        code = tnr_emit(&req, ws, ws_bytes, &o, stream, err, kErrLen);
        if (code != TNR_OK) return failed(code);
    }
    wait();
    int64_t count = 0;
    code = tnr_count_finish(words, &count, err, kErrLen);
    const bool retried = code == TNR_RETRY;
    if (retried) {
        // the hint did not hold: count again in full; the speculative emit
        // wrote nothing
        code = tnr_count_async(&req, ws, ws_bytes, words, stream, err, kErrLen);
        if (code != TNR_OK) return failed(code);
        record();
        wait();
        code = tnr_count_finish(words, &count, err, kErrLen);
    }
    if (code != TNR_OK) return failed(code);
    const int64_t plan = words[3], bins = words[4], mask_need = words[5];
    if (!want.empty()) {
        const bool emitted = reserved == kMissed;
        bool fits = false;
        if (emitted) {
            // the speculative emit covered the count's kernel families (bits
            // 0-1), took the molecule kernel (bit 2) only if every
            // brute-force structure is still a molecule, and launched enough
            // cell-list workgroups
            const int64_t plan_guess = std::get<1>(*guess), bins_guess = std::get<2>(*guess);
            fits = !retried && count <= rows && (plan & ~plan_guess & 3) == 0 &&
                   (!(plan & 1) || !(plan_guess & 4) || (plan & 4)) &&
                   (!(plan & 2) || bins <= bins_guess);
            if (fits) reserved = kFitted;
        }
        if (!emitted || count > rows) {
            rows = count;
            out = Rows{};
            out.allocate(want, rows, pos);
        }
        if (!fits && count > 0) {
            const tnr_outputs o = out.outputs(count, plan, bins);
            code = tnr_emit(&req, ws, ws_bytes, &o, stream, err, kErrLen);
            if (code != TNR_OK) return failed(code);
        }
        out.trim(count, rows);
    }
    if (need_grad) {
        std::optional<Tensor> runs;
        if (sorted && (plan & 3) == 2 && count >= run_pairs && req.n_atoms > run_atoms) {
            runs = at::empty({req.n_atoms, 2}, pos.options().dtype(at::kLong));
            code = tnr_source_runs(&req, ws, ws_bytes, runs->data_ptr(), stream, err, kErrLen);
            if (code != TNR_OK) return failed(code);
        }
        std::tie(*out.D, out.d) =
            fused_geometry(positions, cell, *out.P, *out.S, bp, *out.D, out.d, runs);
    }
    std::vector<Tensor> result;
    result.reserve(quantities.size());
    for (const char c : quantities) result.push_back(out.get(c));
    return Answer{TNR_OK, std::string(), std::move(result), Guess{count, plan, bins, mask_need},
                  reserved};
}

}  // namespace

// Both run without the GIL, as torch's own functions do: an allocation that
// waits for the device, a full launch queue or the wait for the count leaves
// the other Python threads running.  (Saved-tensor hooks take it themselves.)
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    // what the loader compares (tonari_amd/_extensions.py, check_native)
    m.attr("abi_version") = TNR_ABI_VERSION;
    m.attr("torch_version") =
        std::to_string(TORCH_VERSION_MAJOR) + "." + std::to_string(TORCH_VERSION_MINOR);
    m.def("search", [](const std::string& quantities, const Tensor& positions, const Tensor& cell,
                       const Tensor& pbc, const Tensor& batch_ptr, double cutoff,
                       int64_t algorithm, bool sorted, bool half_list, bool include_self,
                       bool need_grad, const std::optional<Guess>& guess, int64_t host,
                       int64_t event, int64_t run_pairs, int64_t run_atoms) {
        HANDLE_TH_ERRORS
        pybind11::gil_scoped_release no_gil;
        return search(quantities, positions, cell, pbc, batch_ptr, cutoff, algorithm, sorted,
                      half_list, include_self, need_grad, guess, host, event, run_pairs, run_atoms);
        END_HANDLE_TH_ERRORS_PYBIND
    });
    m.def("fused_geometry",
          [](const Tensor& positions, const Tensor& cell, const Tensor& pairs,
             const Tensor& shifts, const Tensor& batch_ptr, const Tensor& vectors,
             const std::optional<Tensor>& distances, const std::optional<Tensor>& runs) {
              HANDLE_TH_ERRORS
              pybind11::gil_scoped_release no_gil;
              return fused_geometry(positions, cell, pairs, shifts, batch_ptr, vectors, distances,
                                    runs);
              END_HANDLE_TH_ERRORS_PYBIND
          });
}

// PyTorch C++ extension for the operator (end2end/spatha_mod/block_sparse/api/spatha.cu:41-65 in the reference:
// `spmm(A_metadata, A_indices, A_values, rhs_matrix, bias, A_num_rows, A_num_cols, B_num_cols, vec_length, n, m, nnz,
// seed, mbrow, brow) -> Tensor`, bound with pybind11 under the name `spmm`).  Same argument order and meaning; the work
// itself goes through the C ABI of include/spatha.h on torch's current HIP stream.  Written against the ROCm build of
// PyTorch directly (c10/hip, ATen/hip), not passed through a source translator.
//
// The reference packs nothing per call (its kernel reads the canonical arrays); here the derived operand copies live
// in a plan, so the extension keeps a cache of plans keyed by the identity and version of the three weight tensors.
// An entry holds the tensors, so an address cannot be recycled under a stale plan.  A plan is held through a shared_ptr whose
// deleter destroys it: a launch keeps its own reference, so an eviction or clear_plan_cache() from another thread cannot
// free the plan's device buffers under a launch that is being enqueued.  An in-place update of the weights bumps the tensors'
// version: the miss that follows drops the entries of the same three addresses with an older version, so a loop that
// re-sparsifies in place keeps one plan per matrix.  A write that torch does not see (through `.data` or a raw pointer)
// leaves the version alone: call invalidate_plans(values) or clear_plan_cache() after one.

#include <torch/extension.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/python_variable.h>

#include <list>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <tuple>
#include <unordered_map>

#include "../../include/spatha.h"

namespace {

struct PlanKey {
    const void *values, *metadata, *columns;
    uint32_t v_values, v_metadata, v_columns;
    int rows, cols, n, m, v, device;
    bool operator==(const PlanKey& o) const {
        return values == o.values && metadata == o.metadata && columns == o.columns && v_values == o.v_values &&
               v_metadata == o.v_metadata && v_columns == o.v_columns && rows == o.rows && cols == o.cols && n == o.n &&
               m == o.m && v == o.v && device == o.device;
    }
};
struct PlanKeyHash {
    size_t operator()(const PlanKey& k) const {
        size_t h = std::hash<const void*>()(k.values);
        auto mix = [&h](size_t x) { h ^= x + 0x9e3779b97f4a7c15ull + (h << 6) + (h >> 2); };
        mix(std::hash<const void*>()(k.metadata));
        mix(std::hash<const void*>()(k.columns));
        mix(((size_t)k.v_values << 32) ^ ((size_t)k.v_metadata << 16) ^ k.v_columns);
        mix(((size_t)k.rows << 32) ^ (size_t)k.cols);
        mix(((size_t)k.m << 40) ^ ((size_t)k.v << 20) ^ ((size_t)k.n << 8) ^ (size_t)k.device);
        return h;
    }
};
struct PlanEntry {
    PlanKey key;
    std::shared_ptr<spatha_spmm_plan> plan;
    torch::Tensor values, metadata, columns;      // kept alive for the plan's lifetime
};

constexpr size_t kMaxPlans = 1024;
std::mutex g_lock;
std::list<PlanEntry> g_lru;                                                           // most recently used first
std::unordered_map<PlanKey, std::list<PlanEntry>::iterator, PlanKeyHash> g_index;

void check(int status, const char* what) {
    if (status != SPATHA_OK)
        throw std::runtime_error(std::string(what) + ": " + spatha_status_string(status) +
                                 (status == SPATHA_ERR_HIP ? " (HIP error " + std::to_string(spatha_last_hip_error()) + ")" : ""));
}

// The capture that records what is issued to `stream` now, 0 where nothing records it.
unsigned long long capture_of(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) (void)hipGetLastError();
    return status == hipStreamCaptureStatusActive ? id : 0ull;
}

// Scratch memory of split runs (spatha_spmm_run_ws): one zero-initialised buffer per (device, stream), grown on demand.
// Calls on one stream are ordered, so they can share it; the library leaves it clean after every completed call.
// A buffer made while a graph is captured is not kept: its zeros are written by the graph's replays only.
std::map<std::pair<int, hipStream_t>, torch::Tensor> g_workspaces;

torch::Tensor workspace_for(int device, hipStream_t stream, size_t bytes, const torch::TensorOptions& like) {
    std::lock_guard<std::mutex> guard(g_lock);
    const auto kept = g_workspaces.find({device, stream});
    if (kept != g_workspaces.end() && (size_t)kept->second.numel() >= bytes) return kept->second;
    const torch::Tensor ws = torch::zeros({(int64_t)bytes}, like.dtype(torch::kUInt8));
    if (!capture_of(stream)) g_workspaces[{device, stream}] = ws;
    return ws;
}

void check_weight(const torch::Tensor& t, c10::ScalarType a, c10::ScalarType b, const char* name) {
    TORCH_CHECK(t.is_cuda(), name, " must live on the GPU");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
    TORCH_CHECK(t.scalar_type() == a || t.scalar_type() == b, name, " has the wrong dtype");
}

uint32_t version_of(const torch::Tensor& t) { return (uint32_t)t.unsafeGetTensorImpl()->version_counter().current_version(); }

bool same_storage(const PlanKey& a, const PlanKey& b) {
    return a.values == b.values && a.metadata == b.metadata && a.columns == b.columns && a.device == b.device;
}

// (g_lock held) drops every entry for which `stale` holds; launches that still hold a reference keep their plan alive
template <class Pred>
void drop_entries(Pred stale) {
    for (auto it = g_lru.begin(); it != g_lru.end();) {
        if (stale(*it)) {
            g_index.erase(it->key);
            it = g_lru.erase(it);
        } else {
            ++it;
        }
    }
}

std::shared_ptr<spatha_spmm_plan> plan_for(const torch::Tensor& values, const torch::Tensor& metadata, const torch::Tensor& columns, int rows,
                           int cols, int n, int m, int v, hipStream_t stream) {
    PlanKey key{values.data_ptr(), metadata.data_ptr(), columns.data_ptr(), version_of(values), version_of(metadata),
                version_of(columns), rows, cols, n, m, v, (int)values.get_device()};
    std::lock_guard<std::mutex> guard(g_lock);
    auto hit = g_index.find(key);
    if (hit != g_index.end()) {
        g_lru.splice(g_lru.begin(), g_lru, hit->second);
        return hit->second->plan;
    }
    spatha_spmm_plan* raw = nullptr;
    check(spatha_spmm_plan_create(rows, cols, n, m, v, (const uint16_t*)values.data_ptr(), (const uint32_t*)metadata.data_ptr(),
                                  (const uint32_t*)columns.data_ptr(), stream, &raw),
          "spatha_spmm_plan_create");
    std::shared_ptr<spatha_spmm_plan> plan(raw, [](spatha_spmm_plan* p) { spatha_spmm_plan_destroy(p); });
    // the same three tensors at another version: the weights were rewritten in place, those plans are stale
    drop_entries([&key](const PlanEntry& e) { return same_storage(e.key, key); });
    g_lru.push_front(PlanEntry{key, plan, values.detach(), metadata, columns});
    g_index[key] = g_lru.begin();
    while (g_lru.size() > kMaxPlans) {
        g_index.erase(g_lru.back().key);
        g_lru.pop_back();
    }
    return plan;
}

// memory of its own: no subclass that dispatches to Python and none of functorch's wrappers
bool plain(const torch::Tensor& t) {
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                           c10::DispatchKey::Functionalize});
    return !t.key_set().has_any(wrapped);
}

bool weight_ok(const torch::Tensor& t, c10::ScalarType type, int device) {
    return t.defined() && plain(t) && t.is_cuda() && t.get_device() == device && t.scalar_type() == type && t.is_contiguous();
}

// The V:N:M arrays of a matrix in order on the GPU, magnitude selection and encoding: (values, metadata, columns), or None for what the
// general path decides, and refuses.
py::object convert(py::handle input, int n, int m, int v) {
    if (!THPVariable_CheckExact(input.ptr())) return py::none();
    const torch::Tensor& x = THPVariable_Unpack(input.ptr());
    if (!x.is_cuda() || x.layout() != torch::kStrided || x.dim() != 2 || x.numel() == 0 || !x.is_contiguous() || x.size(0) > INT32_MAX ||
        x.size(1) > INT32_MAX || (x.scalar_type() != torch::kFloat16 && x.scalar_type() != torch::kFloat32))
        return py::none();
    spatha_vnm_geometry geo;
    const int rows = (int)x.size(0), cols = (int)x.size(1);
    if (spatha_vnm_geometry_init(rows, cols, n, m, v, &geo) != SPATHA_OK) return py::none();
    const torch::NoGradGuard no_grad;
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(x.device());
    const torch::TensorOptions on = torch::TensorOptions().device(x.device());
    torch::Tensor values = torch::empty({geo.n_values}, on.dtype(torch::kFloat16)), metadata = torch::empty({geo.n_metadata}, on.dtype(torch::kInt32)),
                  columns = torch::empty({geo.n_columns}, on.dtype(torch::kInt32));
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.get_device()).stream();
    if (spatha_vnm_convert_gpu(x.data_ptr(), x.scalar_type() == torch::kFloat16 ? 16 : 32, rows, cols, n, m, v, (uint16_t*)values.data_ptr(),
                               (uint32_t*)metadata.data_ptr(), (uint32_t*)columns.data_ptr(), stream) != SPATHA_OK)
        return py::none();
    auto wrap = [](const torch::Tensor& t) { return py::reinterpret_steal<py::object>(THPVariable_Wrap(t)); };
    return py::make_tuple(wrap(values), wrap(metadata), wrap(columns));
}

// The dense fp16 matrix [rows, cols] of arrays in order on the GPU, complete on return; None for arrays that the kernel does not take, a
// status where a column offset has no place in its group.
py::object to_dense(py::handle values_h, py::handle metadata_h, py::handle columns_h, int rows, int cols, int n, int m, int v) {
    if (!THPVariable_CheckExact(values_h.ptr()) || !THPVariable_CheckExact(metadata_h.ptr()) || !THPVariable_CheckExact(columns_h.ptr()))
        return py::none();
    const torch::Tensor &values = THPVariable_Unpack(values_h.ptr()), &metadata = THPVariable_Unpack(metadata_h.ptr()),
                        &columns = THPVariable_Unpack(columns_h.ptr());
    if (!values.is_cuda()) return py::none();
    const int device = (int)values.get_device();
    spatha_vnm_geometry geo;
    if (spatha_vnm_geometry_init(rows, cols, n, m, v, &geo) != SPATHA_OK || !weight_ok(values, torch::kFloat16, device) ||
        !weight_ok(metadata, torch::kInt32, device) || !weight_ok(columns, torch::kInt32, device) || values.numel() != geo.n_values ||
        metadata.numel() != geo.n_metadata || columns.numel() != geo.n_columns ||
        (((uintptr_t)values.data_ptr() | (uintptr_t)metadata.data_ptr() | (uintptr_t)columns.data_ptr()) & 3u))
        return py::none();
    const torch::NoGradGuard no_grad;
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(values.device());
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
    torch::Tensor dense = torch::empty({rows, cols}, torch::TensorOptions().device(values.device()).dtype(torch::kFloat16));
    torch::Tensor flag = torch::empty({1}, torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true));
    volatile int* bad = flag.data_ptr<int>();
    *bad = 0;
    check(spatha_vnm_decode_f16_gpu((const uint16_t*)values.data_ptr(), (const uint32_t*)metadata.data_ptr(), (const uint32_t*)columns.data_ptr(),
                                    rows, cols, n, m, v, (uint16_t*)dense.data_ptr(), (uint32_t*)flag.data_ptr(), stream),
          "spatha_vnm_decode");
    {
        const py::gil_scoped_release release;
        const hipError_t e = hipStreamSynchronize(stream);
        if (e != hipSuccess) throw std::runtime_error(std::string("spatha_vnm_decode: ") + hipGetErrorString(e));
    }
    if (*bad) return py::int_((int)SPATHA_ERR_BAD_ARGUMENT);
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(dense));
}

// x [rows, columns], contiguous, with zero columns up to the next multiple of 8
torch::Tensor pad_columns(const torch::Tensor& x) {
    const int64_t columns = x.size(1);
    torch::Tensor out = torch::empty({x.size(0), (columns + 7) / 8 * 8}, x.options().requires_grad(false));
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.get_device()).stream();
    check(spatha_pad_columns_f16((const uint16_t*)x.data_ptr(), (int)x.size(0), (int)columns, (uint16_t*)out.data_ptr(), stream),
          "spatha_pad_columns_f16");
    return out;
}

// full [rows, columns padded to a multiple of 8] -> [rows, columns], contiguous
torch::Tensor cut_columns(const torch::Tensor& full, int64_t columns) {
    torch::Tensor out = torch::empty({full.size(0), columns}, full.options().requires_grad(false));
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(full.get_device()).stream();
    check(spatha_cut_columns_f16((const uint16_t*)full.data_ptr(), (int)full.size(0), (int)columns, (uint16_t*)out.data_ptr(), stream),
          "spatha_cut_columns_f16");
    return out;
}

// The product on a right-hand side of any number of columns where a kernel is chosen that takes it, from rhs as it lies or a padded copy;
// else an undefined tensor, and `padded` holds the copy for the caller's product.  status: of that kernel's run, which may be a refusal.
torch::Tensor run_ragged(const spatha_spmm_plan* plan, const torch::Tensor& rhs, const uint16_t* bias_ptr, int rows, bool transposed_out,
                         int activation, bool fused, torch::Tensor& padded, int& status) {
    status = SPATHA_OK;
    const int tokens = (int)rhs.size(1), layout = transposed_out ? SPATHA_OUT_TRANSPOSED : SPATHA_OUT_ROW_MAJOR;
    const int route = spatha_spmm_ragged_route(plan, tokens, layout, activation != SPATHA_ACT_NONE || (!transposed_out && bias_ptr) ? 1 : 0);
    const bool as_it_lies = route == 2 && ((uintptr_t)rhs.data_ptr() & 15) == 0;
    if (!as_it_lies) padded = pad_columns(rhs);
    if (route == 0) return torch::Tensor();
    const torch::Tensor& B = as_it_lies ? rhs : padded;
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(rhs.get_device()).stream();
    torch::Tensor out = transposed_out ? torch::empty({tokens, rows}, rhs.options().requires_grad(false))
                                       : torch::empty({rows, tokens}, rhs.options().requires_grad(false));
    status = spatha_spmm_run_ragged(plan, (const uint16_t*)B.data_ptr(), (int)B.size(1), tokens, bias_ptr, (uint16_t*)out.data_ptr(), layout,
                                    activation, fused ? 1 : 0, stream);
    return out;
}

// the product on a right-hand side [cols, tokens], tokens a multiple of 8, with operands that have been checked
torch::Tensor run_full(const torch::Tensor& A_metadata, const torch::Tensor& A_indices, const torch::Tensor& A_values,
                       const torch::Tensor& rhs, int tokens, const uint16_t* bias_ptr, int rows, int cols, int v, int n, int m,
                       bool transposed_out, int activation, bool fused, bool read_next = false) {
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(A_values.get_device()).stream();
    // (this reference outlives the launch calls below, whatever another thread does to the cache meanwhile)
    const std::shared_ptr<spatha_spmm_plan> plan = plan_for(A_values, A_metadata, A_indices, rows, cols, n, m, v, stream);
    torch::Tensor out = transposed_out ? torch::empty({tokens, rows}, rhs.options().requires_grad(false))
                                       : torch::empty({rows, tokens}, rhs.options().requires_grad(false));
    const int layout = transposed_out ? SPATHA_OUT_TRANSPOSED : SPATHA_OUT_ROW_MAJOR;
    // few tokens against a long k-loop: the library splits the k-loops over workgroups if it is given scratch memory
    const bool fuses = fused && (activation != SPATHA_ACT_NONE || (!transposed_out && bias_ptr));
    torch::Tensor ws;
    if (const size_t need = spatha_spmm_workspace_bytes(plan.get(), tokens, layout, fuses ? 1 : 0))
        ws = workspace_for((int)A_values.get_device(), stream, need, rhs.options());
    if (read_next) {
        check(spatha_spmm_run_layer(plan.get(), (const uint16_t*)rhs.data_ptr(), tokens, bias_ptr, (uint16_t*)out.data_ptr(), layout,
                                    fused ? activation : SPATHA_ACT_NONE, ws.defined() ? ws.data_ptr() : nullptr,
                                    ws.defined() ? (size_t)ws.numel() : 0, stream),
              "spatha_spmm_run_layer");
        return out;
    }
    if (ws.defined()) {
        check(spatha_spmm_run_ws(plan.get(), (const uint16_t*)rhs.data_ptr(), tokens, bias_ptr, (uint16_t*)out.data_ptr(), layout,
                                 fused ? activation : SPATHA_ACT_NONE, ws.data_ptr(), (size_t)ws.numel(), stream),
              "spatha_spmm_run_ws");
        return out;
    }
    if (fused)
        check(spatha_spmm_run_fused(plan.get(), (const uint16_t*)rhs.data_ptr(), tokens, bias_ptr, (uint16_t*)out.data_ptr(), layout,
                                    activation, 0, stream),
              "spatha_spmm_run_fused");
    else
        check(spatha_spmm_run(plan.get(), (const uint16_t*)rhs.data_ptr(), tokens, bias_ptr, (uint16_t*)out.data_ptr(), layout, 0,
                              stream),
              "spatha_spmm_run");
    return out;
}

torch::Tensor run(const torch::Tensor& A_metadata, const torch::Tensor& A_indices, const torch::Tensor& A_values,
                  const torch::Tensor& rhs_matrix, const c10::optional<torch::Tensor>& bias, int rows, int cols, int v, int n, int m,
                  bool transposed_out, int activation, bool fused) {
    check_weight(A_values, torch::kFloat16, torch::kFloat16, "A_values");
    check_weight(A_metadata, torch::kInt32, torch::kInt32, "A_metadata");
    check_weight(A_indices, torch::kInt32, torch::kInt32, "A_indices");
    check_weight(rhs_matrix, torch::kFloat16, torch::kFloat16, "rhs_matrix");
    TORCH_CHECK(rhs_matrix.dim() == 2 && rhs_matrix.size(0) == cols, "rhs_matrix must be [A_num_cols, tokens]");
    TORCH_CHECK(rhs_matrix.get_device() == A_values.get_device(), "operands live on different devices");
    const uint16_t* bias_ptr = nullptr;
    if (bias.has_value() && bias->defined()) {
        check_weight(*bias, torch::kFloat16, torch::kFloat16, "bias");
        TORCH_CHECK(bias->numel() == rows, "bias must have A_num_rows elements");
        bias_ptr = (const uint16_t*)bias->data_ptr();
    }
    const int tokens = (int)rhs_matrix.size(1);
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(A_values.device());
    if (tokens % 8 != 0 && tokens > 0) {
        // Most kernels move rows of B and C in 16-byte pieces: where one of those is chosen, a token count that is no multiple of 8
        // runs on a copy of rhs_matrix with zero columns appended, and the result is cut back (the appended columns give
        // bias-only rows / columns, which are dropped).
        hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(A_values.get_device()).stream();
        const std::shared_ptr<spatha_spmm_plan> plan = plan_for(A_values, A_metadata, A_indices, rows, cols, n, m, v, stream);
        int status;
        torch::Tensor padded, out = run_ragged(plan.get(), rhs_matrix, bias_ptr, rows, transposed_out, fused ? activation : SPATHA_ACT_NONE,
                                               fused, padded, status);
        check(status, "spatha_spmm_run_ragged");
        if (out.defined()) return out;
        torch::Tensor full = run_full(A_metadata, A_indices, A_values, padded, (int)padded.size(1), bias_ptr, rows, cols, v, n, m,
                                      transposed_out, activation, fused, !transposed_out);
        return transposed_out ? full.narrow(0, 0, tokens) : cut_columns(full, tokens);
    }
    return run_full(A_metadata, A_indices, A_values, rhs_matrix, tokens, bias_ptr, rows, cols, v, n, m, transposed_out, activation, fused);
}

// x [rows, columns], contiguous -> [columns, rows] in rows padded with zeros to a multiple of 8
torch::Tensor transposed_padded(const torch::Tensor& x) {
    torch::Tensor out = torch::empty({x.size(1), (x.size(0) + 7) / 8 * 8}, x.options().requires_grad(false));
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.get_device()).stream();
    check(spatha_transpose_padded_f16((const uint16_t*)x.data_ptr(), (int)x.size(0), (int)x.size(1), (uint16_t*)out.data_ptr(), stream),
          "spatha_transpose_padded_f16");
    return out;
}

// spatha.transpose for an operand in order; None where the caller's checks have to speak
py::object transpose_f16(py::handle input) {
    if (!THPVariable_CheckExact(input.ptr())) return py::none();
    const torch::Tensor& x = THPVariable_Unpack(input.ptr());
    if (!x.is_cuda() || x.layout() != torch::kStrided || x.scalar_type() != torch::kFloat16 || x.dim() != 2 || !x.is_contiguous() ||
        x.numel() == 0 || x.size(0) % 8 != 0 || x.size(0) > 65535 * 64 || x.size(1) > INT32_MAX || ((uintptr_t)x.data_ptr() & 15))
        return py::none();
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(x.device());
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(transposed_padded(x)));
}

// Where work issued now on torch's current stream of `device` runs: the stream, and the capture that records it (0: none).  What one
// call has computed may be taken by a later one only from the same place: another stream is not ordered behind it, a graph replays
// only what was recorded into it, and what was recorded has not run.
py::tuple stream_key(int device) {
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
    return py::make_tuple((uintptr_t)stream, capture_of(stream));
}

// Is `key` the Python key (address, shape, strides, version, device, stream_key) of `held`, and is x the same tensor at the same
// version, used in the same place?
bool same_activation(const torch::Tensor& x, const torch::Tensor& held, const py::tuple& key, const py::tuple& place) {
    return x.data_ptr() == held.data_ptr() && x.sizes() == held.sizes() && x.strides() == held.strides() && x.device() == held.device() &&
           key.size() == 6 && key[3].cast<int64_t>() == (int64_t)x._version() && place.equal(key[5]);
}

// One V:N:M layer on x [..., cols], without a trip through Python per part: the right-hand side (x feature-major already, the
// copy that `last` = (key, activation, copy) holds for this activation, or a new one with padded rows) and the product.  Returns
// (result, new `last` or None), or None for a call this function does not take - the caller's general path decides, and refuses,
// as ever.  feature_major: act(x W^T + b) as a [..., rows] view of a buffer [rows, tokens padded to a multiple of 8], which the
// next layer reads as it lies; else x W^T + b as [..., rows], activation ignored.  transpose: makes the copy where no padding is
// needed (spatha.transpose).
py::object layer_spmm(py::handle input, py::tuple last, const torch::Tensor& metadata, const torch::Tensor& columns,
                      const torch::Tensor& values, const c10::optional<torch::Tensor>& bias, int rows, int cols, int v, int n, int m,
                      bool feature_major, int activation, py::handle transpose) {
    if (!THPVariable_CheckExact(input.ptr())) return py::none();
    const torch::Tensor& x = THPVariable_Unpack(input.ptr());
    if (!x.is_cuda() || x.layout() != torch::kStrided || x.scalar_type() != torch::kFloat16 || x.dim() < 2 || x.size(-1) != cols ||
        x.numel() == 0 || x.is_inference())
        return py::none();
    const int device = (int)x.get_device();
    if (!weight_ok(values, torch::kFloat16, device) || !weight_ok(metadata, torch::kInt32, device) ||
        !weight_ok(columns, torch::kInt32, device) || values.is_inference())
        return py::none();
    const int64_t tokens = x.numel() / cols, padded = (tokens + 7) / 8 * 8;
    if (tokens > 65535 * 64) return py::none();
    const torch::NoGradGuard no_grad;
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(x.device());
    torch::Tensor bias_t;
    if (bias.has_value() && bias->defined()) {
        if (!weight_ok(*bias, torch::kFloat16, device) || bias->numel() != rows) return py::none();
        bias_t = *bias;
    } else if (!feature_major) {
        bias_t = torch::zeros({rows}, x.options().requires_grad(false));
    }
    const torch::Tensor flat = x.dim() == 2 ? x : x.flatten(0, -2);
    auto result = [&](torch::Tensor out, py::object kept) -> py::object {        // out: [tokens, rows] in whatever strides
        if (x.dim() != 2) {
            std::vector<int64_t> sizes(x.sizes().begin(), x.sizes().end());
            sizes.back() = rows;
            out = out.reshape(sizes);
        }
        return py::make_tuple(py::reinterpret_steal<py::object>(THPVariable_Wrap(out)), kept);
    };
    if (!feature_major && tokens <= 16 && flat.is_contiguous() && ((uintptr_t)flat.data_ptr() & 15) == 0) {
        // a few tokens: the kernel reads them as they lie
        hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
        const std::shared_ptr<spatha_spmm_plan> plan = plan_for(values, metadata, columns, rows, cols, n, m, v, stream);
        torch::Tensor out = torch::empty({tokens, rows}, x.options().requires_grad(false));
        const int status = spatha_spmm_run_tokens(plan.get(), (const uint16_t*)flat.data_ptr(), (int)tokens,
                                                  (const uint16_t*)bias_t.data_ptr(), (uint16_t*)out.data_ptr(), stream);
        if (status != SPATHA_ERR_UNSUPPORTED) {
            check(status, "spatha_spmm_run_tokens");
            return result(out, py::none());
        }
    }
    py::object kept = py::none();
    const py::tuple place = stream_key(device);
    torch::Tensor rhs;              // its first element is that of a [cols, padded] matrix
    // [cols, tokens] with rows `pitch` apart, all in memory, readable in 16-byte pieces
    auto holds_padded_rows = [&](const torch::Tensor& t, int64_t pitch) {
        return pitch == padded && (size_t)((t.storage_offset() + cols * padded) * 2) <= t.storage().nbytes() &&
               ((uintptr_t)t.data_ptr() & 15) == 0;
    };
    if (flat.stride(0) == 1 && flat.stride(1) >= tokens && holds_padded_rows(flat, flat.stride(1))) {
        rhs = flat;
    } else {
        torch::Tensor copy;
        if (flat.stride(0) == 1 && flat.stride(1) == tokens) {
            copy = flat.t();
        } else if (last.size() == 3 && THPVariable_Check(last[1].ptr()) && THPVariable_Check(last[2].ptr()) &&
                   same_activation(flat, THPVariable_Unpack(last[1].ptr()), last[0].cast<py::tuple>(), place)) {
            copy = THPVariable_Unpack(last[2].ptr());
        } else {
            const torch::Tensor dense = flat.contiguous();
            if ((uintptr_t)dense.data_ptr() & 15) return py::none();
            py::object made;
            if (padded == tokens) {
                made = transpose(py::reinterpret_steal<py::object>(THPVariable_Wrap(dense)));
                if (!THPVariable_Check(made.ptr())) return py::none();
                copy = THPVariable_Unpack(made.ptr());
            } else {
                copy = transposed_padded(dense).narrow(1, 0, tokens);
                made = py::reinterpret_steal<py::object>(THPVariable_Wrap(copy));
            }
            const py::object held = py::reinterpret_steal<py::object>(THPVariable_Wrap(flat));
            py::tuple shape(2), strides(2);
            for (int d = 0; d < 2; d++) {
                shape[d] = py::int_(flat.size(d));
                strides[d] = py::int_(flat.stride(d));
            }
            kept = py::make_tuple(py::make_tuple(py::int_((uintptr_t)flat.data_ptr()), shape, strides, py::int_((int64_t)flat._version()),
                                                 held.attr("device"), place),
                                  held, made);
        }
        if (copy.dim() != 2 || copy.size(0) != cols || copy.size(1) != tokens || copy.scalar_type() != torch::kFloat16) return py::none();
        if (copy.stride(1) == 1 && holds_padded_rows(copy, copy.stride(0))) rhs = copy;
        else if (padded == tokens && ((uintptr_t)copy.data_ptr() & 15)) return py::none();       // the operator refuses the address
        else rhs = pad_columns(copy.contiguous());
    }
    const uint16_t* bias_ptr = bias_t.defined() ? (const uint16_t*)bias_t.data_ptr() : nullptr;
    torch::Tensor out = run_full(metadata, columns, values, rhs, (int)padded, bias_ptr, rows, cols, v, n, m, !feature_major,
                                 feature_major ? activation : SPATHA_ACT_NONE, feature_major, true);
    if (padded != tokens) out = out.narrow(feature_major ? 1 : 0, 0, tokens);
    return result(feature_major ? out.t() : out, kept);
}

// The attention of `heads` heads of 64 features over qkv [batch * seq, 3 * heads * 64] (queries, keys, values side by side): [batch, seq,
// heads * 64] as a view of a feature-major buffer, which the output projection reads as it lies.  None for an operand that the
// kernel does not take.
py::object attention(py::handle input, int64_t batch, int64_t seq, int64_t heads, double scale) {
    if (!THPVariable_CheckExact(input.ptr())) return py::none();
    const torch::Tensor& qkv = THPVariable_Unpack(input.ptr());
    const int64_t tokens = batch * seq, hidden = heads * 64, padded = (tokens + 7) / 8 * 8;
    if (!qkv.is_cuda() || qkv.layout() != torch::kStrided || qkv.scalar_type() != torch::kFloat16 || qkv.dim() != 2 || batch <= 0 || seq <= 0 ||
        heads <= 0 || qkv.size(0) != tokens || qkv.size(1) != 3 * hidden || !qkv.is_contiguous() || ((uintptr_t)qkv.data_ptr() & 15) ||
        tokens > INT32_MAX / 2 || seq > (1 << 20))
        return py::none();
    const torch::NoGradGuard no_grad;
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(qkv.device());
    torch::Tensor out = torch::empty({hidden, padded}, qkv.options().requires_grad(false));
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(qkv.get_device()).stream();
    const uint16_t* q = (const uint16_t*)qkv.data_ptr();
    check(spatha_attention_f16(q, q + hidden, q + 2 * hidden, 3 * hidden, (int)batch, (int)seq, (int)heads, 64, (float)scale,
                               (uint16_t*)out.data_ptr(), padded, stream),
          "spatha_attention_f16");
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(out.narrow(1, 0, tokens).t().view({batch, seq, hidden})));
}

bool row_ok(const torch::Tensor& t, int device, int64_t numel) {
    return weight_ok(t, torch::kFloat16, device) && t.numel() == numel && ((uintptr_t)t.data_ptr() & 15) == 0;
}

// x's outputs of a norm: [..., hidden] and, with feature_major, its copy [hidden, tokens] in rows padded to a multiple of 8 (else undefined)
struct NormOut {
    torch::Tensor out, padded;
    int64_t tokens;
    py::object tuple() const {
        const py::object second = padded.defined() ? py::reinterpret_steal<py::object>(THPVariable_Wrap(padded.narrow(1, 0, tokens))) : py::none();
        return py::make_tuple(py::reinterpret_steal<py::object>(THPVariable_Wrap(out)), second);
    }
};

// LayerNorm(x + residual) of fp16 operands in order: (result, feature-major copy or None), or None for what the general path decides
py::object add_layernorm(py::handle input, py::handle addend, const torch::Tensor& weight, const torch::Tensor& bias, double eps,
                         bool feature_major) {
    if (!THPVariable_CheckExact(input.ptr()) || !THPVariable_CheckExact(addend.ptr())) return py::none();
    const torch::Tensor &x = THPVariable_Unpack(input.ptr()), &r = THPVariable_Unpack(addend.ptr());
    if (!x.is_cuda() || x.layout() != torch::kStrided || x.dim() < 1 || x.numel() == 0) return py::none();
    const int device = (int)x.get_device();
    const int64_t hidden = x.size(-1), tokens = x.numel() / hidden;
    if (!row_ok(x, device, x.numel()) || !row_ok(r, device, x.numel()) || r.sizes() != x.sizes() || !row_ok(weight, device, hidden) ||
        !row_ok(bias, device, hidden) || hidden % 8 != 0 || hidden > 4096 || tokens > INT32_MAX - 64)
        return py::none();
    const torch::NoGradGuard no_grad;
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(x.device());
    NormOut o;
    o.tokens = tokens;
    o.out = torch::empty(x.sizes(), x.options().requires_grad(false));
    if (feature_major) o.padded = torch::empty({hidden, (tokens + 7) / 8 * 8}, x.options().requires_grad(false));
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
    const uint16_t *xp = (const uint16_t*)x.data_ptr(), *rp = (const uint16_t*)r.data_ptr(), *g = (const uint16_t*)weight.data_ptr(),
                   *b = (const uint16_t*)bias.data_ptr();
    if (feature_major)
        check(spatha_add_layernorm_f16_tp(xp, rp, g, b, (float)eps, (int)tokens, (int)hidden, (uint16_t*)o.out.data_ptr(),
                                          (uint16_t*)o.padded.data_ptr(), stream),
              "spatha_add_layernorm_f16_tp");
    else
        check(spatha_add_layernorm_f16(xp, rp, g, b, (float)eps, (int)tokens, (int)hidden, (uint16_t*)o.out.data_ptr(), stream),
              "spatha_add_layernorm_f16");
    return o.tuple();
}

// The embedding of ids [batch, seq]: word, type and position tables, LayerNorm; types [batch, seq] or [1, >= seq] (own_types: the
// model's row of them, looked up at the position ids), positions [1, >= seq].  As add_layernorm.
py::object embed_layernorm(const torch::Tensor& ids, const torch::Tensor& types, const torch::Tensor& positions, const torch::Tensor& word,
                           const torch::Tensor& type, const torch::Tensor& position, const torch::Tensor& weight, const torch::Tensor& bias,
                           double eps, bool feature_major, bool own_types) {
    if (!plain(ids) || !ids.is_cuda() || ids.layout() != torch::kStrided || ids.dim() != 2 || ids.numel() == 0) return py::none();
    // (a tangent of forward-mode differentiation is the stock operations' to carry on)
    for (const torch::Tensor* t : {&word, &type, &position, &weight, &bias})
        if (!plain(*t) || t->_fw_grad(0).defined()) return py::none();
    const int device = (int)ids.get_device();
    const int64_t batch = ids.size(0), seq = ids.size(1), hidden = word.dim() == 2 ? word.size(1) : 0;
    const bool types_shared = types.dim() == 2 && types.size(0) == 1 && types.size(1) >= seq;
    if (!weight_ok(ids, torch::kInt64, device) || !weight_ok(types, torch::kInt64, device) || !weight_ok(positions, torch::kInt64, device) ||
        !(types_shared || (!own_types && types.sizes() == ids.sizes())) || positions.dim() != 2 || positions.size(0) != 1 || positions.size(1) < seq ||
        hidden <= 0 || hidden % 8 != 0 || hidden > 4096 || batch * seq > INT32_MAX - 64)
        return py::none();
    for (const torch::Tensor* t : {&word, &type, &position})
        if (t->dim() != 2 || t->size(1) != hidden || t->size(0) <= 0 || !row_ok(*t, device, t->numel())) return py::none();
    if (!row_ok(weight, device, hidden) || !row_ok(bias, device, hidden)) return py::none();
    const torch::NoGradGuard no_grad;
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(ids.device());
    NormOut o;
    o.tokens = batch * seq;
    o.out = torch::empty({batch, seq, hidden}, word.options().requires_grad(false));
    if (feature_major) o.padded = torch::empty({hidden, (o.tokens + 7) / 8 * 8}, word.options().requires_grad(false));
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
    auto* embed = own_types ? &spatha_embed_layernorm_own_types_f16 : &spatha_embed_layernorm_f16;
    check(embed((const int64_t*)ids.data_ptr(), (const int64_t*)types.data_ptr(), own_types ? types.size(1) : types_shared ? 0 : seq,
                (const int64_t*)positions.data_ptr(), (int)batch, (int)seq, (const uint16_t*)word.data_ptr(), word.size(0),
                (const uint16_t*)type.data_ptr(), type.size(0), (const uint16_t*)position.data_ptr(), position.size(0),
                (const uint16_t*)weight.data_ptr(), (const uint16_t*)bias.data_ptr(), (float)eps, (int)hidden,
                (uint16_t*)o.out.data_ptr(), feature_major ? (uint16_t*)o.padded.data_ptr() : nullptr, stream),
          "spatha_embed_layernorm_f16");
    return o.tuple();
}

// SpmmPlan.run without a k-split, for operands in order; None where the caller's checks have to speak.  bias needs the transposed
// layout unless `fused` (an activation, ACT_NONE among them, was named).
py::object plan_run(size_t handle, py::handle rhs, py::handle bias, py::handle out, int rows, int cols, int device, bool transposed_out,
                    bool fused, int activation, int variant) {
    if (!THPVariable_CheckExact(rhs.ptr()) || c10::InferenceMode::is_enabled()) return py::none();
    const torch::Tensor& B = THPVariable_Unpack(rhs.ptr());
    if (!weight_ok(B, torch::kFloat16, device) || B.dim() != 2 || B.size(0) != cols || B.size(1) <= 0 || B.size(1) > INT32_MAX - 8)
        return py::none();
    const bool ragged = B.size(1) % 8 != 0;
    if (ragged && (variant != 0 || !out.is_none())) return py::none();
    const int N = (int)B.size(1);
    const uint16_t* bias_ptr = nullptr;
    if (!bias.is_none()) {
        if (!THPVariable_Check(bias.ptr())) return py::none();
        const torch::Tensor& b = THPVariable_Unpack(bias.ptr());
        if (!weight_ok(b, torch::kFloat16, device) || b.numel() != rows) return py::none();
        bias_ptr = (const uint16_t*)b.data_ptr();
    }
    const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(B.device());
    const spatha_spmm_plan* plan = (const spatha_spmm_plan*)handle;
    if (ragged) {
        if (!fused && !transposed_out && bias_ptr) return py::none();          // (refused)
        const torch::NoGradGuard no_grad;
        int status;
        torch::Tensor padded, got = run_ragged(plan, B, bias_ptr, rows, transposed_out, activation, fused, padded, status);
        if (status != SPATHA_OK) return py::int_(status);
        if (!got.defined()) {
            const int64_t n_padded = padded.size(1);
            got = transposed_out ? torch::empty({n_padded, rows}, B.options().requires_grad(false))
                                 : torch::empty({rows, n_padded}, B.options().requires_grad(false));
            hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
            const uint16_t* b_ptr = (const uint16_t*)padded.data_ptr();
            uint16_t* c_ptr = (uint16_t*)got.data_ptr();
            // (a row-major result is read at once, by the cut)
            status = !transposed_out ? spatha_spmm_run_layer(plan, b_ptr, (int)n_padded, bias_ptr, c_ptr, SPATHA_OUT_ROW_MAJOR, activation,
                                                             nullptr, 0, stream)
                     : fused ? spatha_spmm_run_fused(plan, b_ptr, (int)n_padded, bias_ptr, c_ptr, SPATHA_OUT_TRANSPOSED, activation, 0, stream)
                             : spatha_spmm_run(plan, b_ptr, (int)n_padded, bias_ptr, c_ptr, SPATHA_OUT_TRANSPOSED, 0, stream);
            if (status != SPATHA_OK) return py::int_(status);
            got = transposed_out ? got.narrow(0, 0, N) : cut_columns(got, N);
        }
        return py::reinterpret_steal<py::object>(THPVariable_Wrap(got));
    }
    torch::Tensor C;
    if (out.is_none()) {
        C = transposed_out ? torch::empty({N, rows}, B.options().requires_grad(false)) : torch::empty({rows, N}, B.options().requires_grad(false));
    } else {
        if (!THPVariable_CheckExact(out.ptr())) return py::none();
        C = THPVariable_Unpack(out.ptr());
        if (!weight_ok(C, torch::kFloat16, device) || C.is_inference() || C.dim() != 2 || C.size(0) != (transposed_out ? N : rows) ||
            C.size(1) != (transposed_out ? rows : N))
            return py::none();
    }
    const uint16_t* b_ptr = (const uint16_t*)B.data_ptr();
    uint16_t* c_ptr = (uint16_t*)C.data_ptr();
    const int layout = transposed_out ? SPATHA_OUT_TRANSPOSED : SPATHA_OUT_ROW_MAJOR;
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream();
    int status;
    {
        const py::gil_scoped_release release;
        status = fused ? spatha_spmm_run_fused(plan, b_ptr, N, bias_ptr, c_ptr, layout, activation, variant, stream)
                       : spatha_spmm_run(plan, b_ptr, N, bias_ptr, c_ptr, layout, variant, stream);
    }
    if (status != SPATHA_OK) return py::int_(status);
    // the kernel wrote through a raw pointer: tell torch, so that caches keyed on the tensor's version see the change
    C.unsafeGetTensorImpl()->bump_version();
    if (!out.is_none()) return py::reinterpret_borrow<py::object>(out);
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(C));
}

// out[B_num_cols, A_num_rows] = (A_vnm @ rhs_matrix).T + bias, fp16: the reference operator.  vec_length is V and is
// honoured at run time; nnz and seed are accepted and unused, as there; mbrow / brow must be 32 / 4, the only layout the
// format defines.
torch::Tensor spmm(torch::Tensor A_metadata, torch::Tensor A_indices, torch::Tensor A_values, torch::Tensor rhs_matrix,
                   c10::optional<torch::Tensor> bias, int A_num_rows, int A_num_cols, int B_num_cols, int vec_length, int n, int m,
                   int nnz, int seed, int mbrow, int brow) {
    (void)nnz;
    (void)seed;
    TORCH_CHECK(mbrow == 32 && brow == 4, "only mbrow=32, brow=4 is defined for the V:N:M layout");
    TORCH_CHECK(rhs_matrix.dim() == 2 && rhs_matrix.size(1) == B_num_cols, "B_num_cols does not match rhs_matrix");
    return run(A_metadata, A_indices, A_values, rhs_matrix, bias, A_num_rows, A_num_cols, vec_length, n, m, true, SPATHA_ACT_NONE,
               false);
}

// act((A_vnm @ rhs_matrix) + bias) as [A_num_rows, tokens] (ready to be the rhs of the next spmm) or, with
// transposed_out, as [tokens, A_num_rows]; activation: 0 none, 1 GELU (erf), 2 GELU (tanh)
torch::Tensor spmm_fused(torch::Tensor A_metadata, torch::Tensor A_indices, torch::Tensor A_values, torch::Tensor rhs_matrix,
                         c10::optional<torch::Tensor> bias, int A_num_rows, int A_num_cols, int vec_length, int n, int m,
                         int activation, bool transposed_out) {
    return run(A_metadata, A_indices, A_values, rhs_matrix, bias, A_num_rows, A_num_cols, vec_length, n, m, transposed_out,
               activation, true);
}

void clear_plan_cache() {
    std::lock_guard<std::mutex> guard(g_lock);
    g_lru.clear();
    g_index.clear();
    g_workspaces.clear();
}

// Drops the plans built from this values tensor (any version): for weights changed behind torch's back.
int64_t invalidate_plans(const torch::Tensor& A_values) {
    std::lock_guard<std::mutex> guard(g_lock);
    const size_t before = g_lru.size();
    const void* ptr = A_values.data_ptr();
    drop_entries([ptr](const PlanEntry& e) { return e.key.values == ptr; });
    return (int64_t)(before - g_lru.size());
}

int64_t plan_cache_size() {
    std::lock_guard<std::mutex> guard(g_lock);
    return (int64_t)g_lru.size();
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, mod) {
    mod.def("spmm", &spmm, "V:N:M SpMM: (A_vnm @ rhs).T + bias", py::arg("A_metadata"), py::arg("A_indices"), py::arg("A_values"),
            py::arg("rhs_matrix"), py::arg("bias"), py::arg("A_num_rows"), py::arg("A_num_cols"), py::arg("B_num_cols"),
            py::arg("vec_length"), py::arg("n"), py::arg("m"), py::arg("nnz") = 0, py::arg("seed") = 0, py::arg("mbrow") = 32,
            py::arg("brow") = 4);
    mod.def("spmm_fused", &spmm_fused, "V:N:M SpMM with bias and activation in the write-out", py::arg("A_metadata"),
            py::arg("A_indices"), py::arg("A_values"), py::arg("rhs_matrix"), py::arg("bias"), py::arg("A_num_rows"),
            py::arg("A_num_cols"), py::arg("vec_length"), py::arg("n"), py::arg("m"), py::arg("activation") = 0,
            py::arg("transposed_out") = false);
    mod.def("layer_spmm", &layer_spmm, "one V:N:M layer, right-hand side and product, or None");
    mod.def("attention", &attention, "attention of merged projections, feature-major, or None");
    mod.def("add_layernorm", &add_layernorm, "LayerNorm(x + residual): (result, feature-major copy or None), or None");
    mod.def("embed_layernorm", &embed_layernorm, "LayerNorm of summed table rows: (result, feature-major copy or None), or None");
    mod.def("convert", &convert, "the V:N:M arrays of a matrix on the GPU, or None");
    mod.def("to_dense", &to_dense, "the matrix of V:N:M arrays on the GPU, or None, or the status of a refusal");
    mod.def("stream_key", &stream_key, "(stream, capture) that work issued now on this device goes to", py::arg("device"));
    mod.def("transpose", &transpose_f16, "x.T of an fp16 matrix through the library's kernel, or None");
    mod.def("plan_run", &plan_run, "a plan's product, or None, or the status of a refusal");
    mod.def("clear_plan_cache", &clear_plan_cache, "drop every cached plan");
    mod.def("invalidate_plans", &invalidate_plans, "drop the cached plans built from this values tensor; returns how many",
            py::arg("A_values"));
    mod.def("plan_cache_size", &plan_cache_size, "number of cached plans");
}

// Host side of the calls in native code: argument checks, outputs from torch's
// caching allocator, the current stream, one call of the C ABI.  Host code only
// (no kernels, no GPU run-time calls of its own besides torch's); the kernels and
// every decision about them stay behind include/ash_hip.h, whose functions are
// looked up in the library that the Python loader has opened (`bind`).
//
// A call costs the host 4-6 us this way; the same in Python through ctypes took
// 15-25 us, more than the kernels of a small batch (a find of a thousand keys
// with their rows: 23 us of Python around 7 us of kernel).
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/python_function.h>

#include <dlfcn.h>

#include <memory>
#include <mutex>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/ash_hip.h"

#ifndef ASH_HOST_FINGERPRINT
#define ASH_HOST_FINGERPRINT "unknown"
#endif

namespace {

using torch::Tensor;
namespace py = pybind11;

// --------------------------------------------------------------- the library
#define ASH_FUNCTIONS(X)                                                              \
    X(ash_last_error)                                                                 \
    X(ash_map_find)                                                                   \
    X(ash_map_find_rows_scratch_bytes)                                                \
    X(ash_map_find_rows_scratch)                                                      \
    X(ash_add_rows)                                                                   \
    X(ash_gather_rows)                                                                \
    X(ash_map_insert_scratch_bytes)                                                   \
    X(ash_map_insert_auto)                                                            \
    X(ash_map_clear_rows)                                                             \
    X(ash_map_erase_scratch_bytes)                                                    \
    X(ash_map_erase_auto)                                                             \
    X(ash_map_items)                                                                  \
    X(ash_map_items_rows)                                                             \
    X(ash_map_counters)                                                               \
    X(ash_map_upkeep)                                                                 \
    X(ash_map_neighbors)                                                              \
    X(ash_grid_fuse_frame)                                                            \
    X(ash_ray_volume_bytes)                                                           \
    X(ash_map_ray_volume_bytes)                                                       \
    X(ash_ray_volume_kept)                                                            \
    X(ash_ray_find_near_far_marked)                                                   \
    X(ash_ray_sample_groups)                                                          \
    X(ash_ray_sample_march_marked)                                                    \
    X(ash_ray_sample_place)                                                           \
    X(ash_surface_block8_workspace_bytes)                                             \
    X(ash_surface_block8_classify)                                                    \
    X(ash_surface_block8_extract)                                                     \
    X(ash_grid_query)                                                                 \
    X(ash_grid_forward)                                                               \
    X(ash_query_forward)                                                              \
    X(ash_query_backward_forward)                                                     \
    X(ash_query_backward_forward_scaled)                                              \
    X(ash_query_backward_backward_scaled)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
    ASH_FUNCTIONS(X)
#undef X
} lib;

[[noreturn]] void fail(const std::string& message) { throw std::runtime_error(message); }

void need(bool ok, const char* message) {
    if (!ok) fail(message);
}

void check(int status) {
    if (status != 0) {
        const char* m = lib.ash_last_error();
        fail(m != nullptr && *m ? m : "libash_hip call failed");
    }
}

// `handle`: what dlopen gave the Python loader
void bind(uintptr_t handle) {
    void* h = reinterpret_cast<void*>(handle);
#define X(name)                                                                       \
    lib.name = reinterpret_cast<decltype(&::name)>(dlsym(h, #name));                  \
    if (lib.name == nullptr) fail("libash_hip.so does not export " #name);
    ASH_FUNCTIONS(X)
#undef X
}

// ------------------------------------------------------------------- helpers
ash_map_t* map_of(uintptr_t handle) { return reinterpret_cast<ash_map_t*>(handle); }

void* stream_of(int64_t device) {
    return c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream();
}

Tensor empty(at::IntArrayRef sizes, at::ScalarType type, int64_t device) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(
                                    at::kCUDA, static_cast<c10::DeviceIndex>(device)));
}

// Memory that a call can do without: none where the device has none left.
Tensor scratch_if_there(int64_t bytes, int64_t device) {
    if (bytes <= 0) return Tensor();
    try {
        return empty({bytes}, at::kByte, device);
    } catch (const c10::OutOfMemoryError&) {
        return Tensor();
    }
}

template <typename T>
T* ptr(const Tensor& t) {
    return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}

std::string shape_of(const Tensor& t) {
    std::string s = "(";
    for (int64_t d = 0; d < t.dim(); ++d) {
        s += std::to_string(t.size(d));
        s += d + 1 < t.dim() ? ", " : t.dim() == 1 ? "," : "";
    }
    return s + ")";
}

Tensor keys_of(const Tensor& keys, int64_t dim, int64_t device) {
    if (keys.dim() != 2 || keys.size(1) != dim) {
        fail("keys must be (N, " + std::to_string(dim) + "), got " + shape_of(keys));
    }
    if (!keys.is_cuda() || keys.get_device() != device) {
        fail("keys are on " + keys.device().str() + ", the map on cuda:" + std::to_string(device));
    }
    return keys.to(at::kInt).contiguous();
}

int64_t row_bytes_of(const Tensor& t) {
    return t.numel() / t.size(0) * static_cast<int64_t>(t.element_size());
}

int32_t dtype_of(const Tensor& t, const char* what) {
    if (t.scalar_type() == at::kFloat) return ASH_F32;
    if (t.scalar_type() == at::kDouble) return ASH_F64;
    fail(std::string(what) + " must be float32 or float64, got torch." +
         (t.scalar_type() == at::kHalf ? "float16" : c10::toString(t.scalar_type())));
}

int32_t interpolation_of(const std::string& name) {
    if (name == "linear") return ASH_INTERP_LINEAR;
    if (name == "smooth_step") return ASH_INTERP_SMOOTH_STEP;
    fail("Unknown interpolation functor: " + name);
}

// ------------------------------------------------------------------- look-up
std::tuple<Tensor, Tensor> find(uintptr_t handle, int64_t dim, int64_t device, const Tensor& keys_in) {
    const Tensor keys = keys_of(keys_in, dim, device);
    const int64_t n = keys.size(0);
    Tensor indices = empty({n}, at::kLong, device), masks = empty({n}, at::kBool, device);
    check(lib.ash_map_find(map_of(handle), ptr<int32_t>(keys), n, ptr<int64_t>(indices),
                           ptr<uint8_t>(masks), stream_of(device)));
    return {indices, masks};
}

constexpr int64_t kMaxRowBytes = 32764;   // ash_map_find_rows
constexpr size_t kMaxTables = 4;

bool finds_rows_of(const std::vector<Tensor>& tables, int64_t device) {
    if (tables.empty() || tables.size() > kMaxTables) return false;
    for (const Tensor& t : tables) {
        if (!t.is_cuda() || t.get_device() != device || !t.is_contiguous() || t.dim() < 1 ||
            t.numel() == 0 || t.size(0) > 0x7FFFFFFFll) {
            return false;
        }
        const int64_t bytes = row_bytes_of(t);
        if (bytes > kMaxRowBytes || bytes % 4 != 0) return false;
    }
    return true;
}

std::tuple<Tensor, Tensor, std::vector<Tensor>> find_rows(uintptr_t handle, int64_t dim, int64_t device,
                                                          const Tensor& keys_in,
                                                          const std::vector<Tensor>& tables,
                                                          bool zero_misses, bool need_indices) {
    const Tensor keys = keys_of(keys_in, dim, device);
    need(tables.size() <= kMaxTables, "find_rows takes up to 4 tensors per call");
    const int64_t n = keys.size(0);
    Tensor indices = need_indices ? empty({n}, at::kLong, device) : Tensor();
    Tensor masks = empty({n}, at::kBool, device);
    std::vector<Tensor> rows;
    const void* src[kMaxTables];
    void* dst[kMaxTables];
    int64_t bytes[kMaxTables], count[kMaxTables];
    for (const Tensor& t : tables) {
        const size_t v = rows.size();
        std::vector<int64_t> shape = t.sizes().vec();
        shape[0] = n;
        rows.push_back(empty(shape, t.scalar_type(), device));
        src[v] = t.data_ptr();
        dst[v] = rows[v].data_ptr();
        bytes[v] = row_bytes_of(t);
        count[v] = t.size(0);
    }
    const int n_tables = static_cast<int>(tables.size());
    const Tensor scratch = scratch_if_there(
            lib.ash_map_find_rows_scratch_bytes(map_of(handle), n, n_tables, bytes, count), device);
    check(lib.ash_map_find_rows_scratch(map_of(handle), ptr<int32_t>(keys), n, n_tables, src, dst, bytes,
                                        count, zero_misses, ptr<int64_t>(indices), ptr<uint8_t>(masks),
                                        ptr<void>(scratch), scratch.defined() ? scratch.numel() : 0,
                                        stream_of(device)));
    return {indices, masks, rows};
}

Tensor add_rows(const Tensor& rows_in, const Tensor& indices, const Tensor& masks, int64_t out_rows) {
    need(rows_in.is_cuda() && rows_in.dim() == 2, "rows must be (N, E) on a HIP device");
    const int64_t n = rows_in.size(0), width = rows_in.size(1), device = rows_in.get_device();
    need(indices.numel() == n && masks.numel() == n && indices.scalar_type() == at::kLong &&
                 masks.scalar_type() == at::kBool && indices.is_cuda() && masks.is_cuda() &&
                 indices.get_device() == device && masks.get_device() == device,
         "add_rows: one int64 index and one mask per row are needed");
    const Tensor rows = rows_in.contiguous();
    Tensor out = empty({out_rows, width}, rows.scalar_type(), device);
    check(lib.ash_add_rows(rows.data_ptr(), ptr<int64_t>(indices.contiguous()),
                           ptr<uint8_t>(masks.contiguous()), n, width, dtype_of(rows, "rows"),
                           out.data_ptr(), out_rows, stream_of(device)));
    return out;
}

// Rows of `embedding` under `keys`, zeros for keys that are not stored.  Linear
// in the embedding: its backward (AddRows) and the backward of that need
// nothing but the indices found here.
struct AddRows : torch::autograd::Function<AddRows> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& z, const Tensor& indices,
                          const Tensor& masks, int64_t num_rows) {
        ctx->save_for_backward({indices, masks});
        return add_rows(z, indices, masks, num_rows);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                   torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        return {saved[1].unsqueeze(-1) * grads[0].index({saved[0]}), Tensor(), Tensor(), Tensor()};
    }
};

struct Rows : torch::autograd::Function<Rows> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& embedding,
                          uintptr_t handle, int64_t dim, int64_t device, const Tensor& keys) {
        auto [indices, masks, rows] = find_rows(handle, dim, device, keys, {embedding}, true, true);
        ctx->save_for_backward({indices, masks});
        ctx->saved_data["num_rows"] = embedding.size(0);
        return rows[0];
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                   torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const int64_t num_rows = ctx->saved_data["num_rows"].toInt();
        if (at::globalContext().deterministicAlgorithms()) {
            // add_rows adds by atomics, in any order: where torch is asked for the
            // same numbers on every run, its own backward of indexing, which sorts
            const Tensor rows = saved[1].unsqueeze(-1) * grads[0];
            return {at::zeros({num_rows, rows.size(1)}, rows.options())
                            .index_put({saved[0]}, rows, /*accumulate=*/true),
                    Tensor(), Tensor(), Tensor(), Tensor()};
        }
        Tensor grad = at::GradMode::is_enabled()
                              ? AddRows::apply(grads[0], saved[0], saved[1], num_rows)
                              : add_rows(grads[0], saved[0], saved[1], num_rows);
        return {grad, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

Tensor embedding_rows(const Tensor& embedding, uintptr_t handle, int64_t dim, int64_t device,
                      const Tensor& keys) {
    if (!(at::GradMode::is_enabled() && embedding.requires_grad())) {
        return std::get<2>(find_rows(handle, dim, device, keys, {embedding}, true, false))[0];
    }
    return Rows::apply(embedding, handle, dim, device, keys);
}

// Up to four tables per launch; the first `first` rows where there are no indices.
std::vector<Tensor> gather_rows(const std::vector<Tensor>& tables, const std::optional<Tensor>& indices,
                                int64_t first) {
    std::vector<Tensor> out;
    Tensor index;
    if (indices.has_value()) index = indices->reshape({-1}).contiguous();
    const int64_t n = index.defined() ? index.size(0) : first;
    for (const Tensor& t : tables) {
        std::vector<int64_t> shape = t.sizes().vec();
        shape[0] = n;
        out.push_back(empty(shape, t.scalar_type(), t.get_device()));
    }
    for (size_t start = 0; start < tables.size() && n > 0; start += kMaxTables) {
        const size_t k = std::min(kMaxTables, tables.size() - start);
        const void* src[kMaxTables];
        void* dst[kMaxTables];
        int64_t bytes[kMaxTables], count[kMaxTables];
        for (size_t v = 0; v < k; ++v) {
            const Tensor& t = tables[start + v];
            src[v] = t.data_ptr();
            dst[v] = out[start + v].data_ptr();
            bytes[v] = row_bytes_of(t);
            count[v] = t.size(0);
        }
        check(lib.ash_gather_rows(static_cast<int>(k), src, dst, bytes, count, ptr<int64_t>(index), n,
                                  stream_of(tables[start].get_device())));
    }
    return out;
}

// ----------------------------------------------------------------- mutations
// One ash_map_insert_auto; true: the second region has to be attached and the
// call issued again.
bool insert(uintptr_t handle, int64_t dim, int64_t device, int64_t capacity, const Tensor& keys_in,
            const std::vector<std::string>& names, const std::vector<Tensor>& values,
            const std::vector<Tensor>& stores, int policy) {
    const Tensor keys = keys_of(keys_in, dim, device);
    const int64_t n = keys.size(0);
    const size_t k = names.size();
    std::vector<Tensor> held;
    std::vector<const void*> src;
    std::vector<void*> dst;
    std::vector<int64_t> bytes;
    for (size_t i = 0; i < k; ++i) {
        const Tensor &v = values[i], &ext = stores[i];
        const std::string what = "value '" + names[i] + "'", where = "destination buffer '" + names[i] + "'";
        if (v.dim() < 1 || v.size(0) != n) {
            fail(what + " has " + std::to_string(v.dim() < 1 ? 0 : v.size(0)) + " rows for " +
                 std::to_string(n) + " keys");
        }
        if (v.scalar_type() != ext.scalar_type() || v.sizes().slice(1) != ext.sizes().slice(1)) {
            fail(what + " does not match its destination buffer");
        }
        if (!v.is_cuda() || !ext.is_cuda() || v.get_device() != device || ext.get_device() != device) {
            fail(what + " is not on cuda:" + std::to_string(device));
        }
        if (!ext.is_contiguous()) fail(where + " must be contiguous");
        if (ext.size(0) != capacity) fail(where + " must have `capacity` rows");
        held.push_back(v.contiguous());
        src.push_back(held.back().data_ptr());
        dst.push_back(ext.data_ptr());
        bytes.push_back(n > 0 ? row_bytes_of(v) : 0);
    }
    if (n == 0) return false;
    int64_t scratch_bytes = 0;
    check(lib.ash_map_insert_scratch_bytes(map_of(handle), n, static_cast<int>(k), bytes.data(), policy,
                                           &scratch_bytes));
    const Tensor scratch = scratch_bytes > 0 ? empty({scratch_bytes}, at::kByte, device) : Tensor();
    void* stream = stream_of(device);
    int status;
    {
        py::gil_scoped_release waits_for_the_device;
        status = lib.ash_map_insert_auto(map_of(handle), ptr<int32_t>(keys), n, static_cast<int>(k),
                                         src.data(), dst.data(), bytes.data(), ptr<void>(scratch),
                                         scratch_bytes, policy, nullptr, stream);
    }
    if (status == ASH_NEEDS_GENERAL) return true;
    check(status);
    return false;
}

// Whether the streaming path was taken.
bool erase(uintptr_t handle, int64_t dim, int64_t device, const Tensor& keys_in, int policy) {
    const Tensor keys = keys_of(keys_in, dim, device);
    const int64_t n = keys.size(0);
    int64_t scratch_bytes = 0;
    check(lib.ash_map_erase_scratch_bytes(map_of(handle), n, policy, &scratch_bytes));
    const Tensor scratch = scratch_bytes > 0 ? empty({scratch_bytes}, at::kByte, device) : Tensor();
    check(lib.ash_map_erase_auto(map_of(handle), ptr<int32_t>(keys), n, ptr<void>(scratch), scratch_bytes,
                                 policy, stream_of(device)));
    return scratch_bytes > 0;
}

// What torch's zero_() does to a plain tensor by one fill of its memory.
bool can_zero(const Tensor& t, int64_t device) {
    return t.is_cuda() && t.get_device() == device && t.layout() == at::kStrided && t.is_contiguous() &&
           !t.requires_grad() && !t.is_inference() &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

void clear(uintptr_t handle, int64_t device, const std::vector<Tensor>& zeroed) {
    need(zeroed.size() <= kMaxTables, "clear takes up to 4 tensors per call");
    void* rows[kMaxTables];
    int64_t bytes[kMaxTables];
    for (size_t v = 0; v < zeroed.size(); ++v) {
        need(can_zero(zeroed[v], device), "clear takes contiguous tensors on the map's device");
        rows[v] = zeroed[v].data_ptr();
        bytes[v] = static_cast<int64_t>(zeroed[v].nbytes());
    }
    check(lib.ash_map_clear_rows(map_of(handle), static_cast<int>(zeroed.size()), rows, bytes,
                                 stream_of(device)));
    for (const Tensor& t : zeroed) t.unsafeGetTensorImpl()->bump_version();
}

std::vector<int64_t> counters(uintptr_t handle, int64_t device) {
    std::vector<int64_t> out(7);
    void* stream = stream_of(device);
    int status;
    {
        py::gil_scoped_release waits_for_the_device;
        status = lib.ash_map_counters(map_of(handle), nullptr, out.data(), stream);
    }
    check(status);
    return out;
}

std::tuple<Tensor, Tensor> items(uintptr_t handle, int64_t dim, int64_t device, int64_t n) {
    Tensor keys = empty({n, dim}, at::kInt, device), indices = empty({n}, at::kLong, device);
    if (n > 0) {
        check(lib.ash_map_items(map_of(handle), ptr<int32_t>(keys), ptr<int64_t>(indices), n,
                                stream_of(device)));
    }
    return {keys, indices};
}

std::tuple<Tensor, Tensor, std::vector<Tensor>> items_rows(uintptr_t handle, int64_t dim, int64_t device,
                                                           int64_t n, const std::vector<Tensor>& tables) {
    need(tables.size() <= kMaxTables, "items_rows takes up to 4 tensors per call");
    Tensor keys = empty({n, dim}, at::kInt, device), indices = empty({n}, at::kLong, device);
    std::vector<Tensor> rows;
    const void* src[kMaxTables];
    void* dst[kMaxTables];
    int64_t bytes[kMaxTables], count[kMaxTables];
    for (const Tensor& t : tables) {
        const size_t v = rows.size();
        std::vector<int64_t> shape = t.sizes().vec();
        shape[0] = n;
        rows.push_back(empty(shape, t.scalar_type(), device));
        src[v] = t.data_ptr();
        dst[v] = rows[v].data_ptr();
        bytes[v] = row_bytes_of(t);
        count[v] = t.size(0);
    }
    if (n > 0) {
        check(lib.ash_map_items_rows(map_of(handle), ptr<int32_t>(keys), ptr<int64_t>(indices), n,
                                     static_cast<int>(tables.size()), src, dst, bytes, count,
                                     stream_of(device)));
    }
    return {keys, indices, rows};
}

// (coords (rows, 3), lut (rows, K)) of the keys at offsets within `radius`
std::pair<Tensor, Tensor> neighbors(uintptr_t handle, int64_t device, int64_t rows, int radius,
                                    bool bidirectional) {
    const int64_t width = bidirectional ? 2 * radius + 1 : radius + 1;
    const Tensor coords = empty({rows, 3}, at::kInt, device);
    const Tensor lut = empty({rows, width * width * width}, at::kLong, device);
    check(lib.ash_map_neighbors(map_of(handle), rows, radius, bidirectional, ptr<int32_t>(coords),
                                ptr<int64_t>(lut), stream_of(device)));
    return {coords, lut};
}

// ---------------------------------------------------------------------- grid
Tensor positions_of(const Tensor& x) {
    need(x.dim() == 2 && x.size(1) == 3 && x.scalar_type() == at::kFloat, "positions must be float32 (N, 3)");
    return x.contiguous();
}

std::tuple<Tensor, Tensor, Tensor, Tensor> query_cells(uintptr_t handle, int64_t device, const Tensor& x_in,
                                                       int grid_dim) {
    const Tensor x = positions_of(x_in);
    if (!x.is_cuda() || x.get_device() != device) {
        fail("positions are on " + x.device().str() + ", the map on cuda:" + std::to_string(device));
    }
    const int64_t n = x.size(0);
    Tensor grids = empty({n}, at::kLong, device), cells = empty({n}, at::kLong, device);
    Tensor offsets = empty({n, 3}, at::kFloat, device), masks = empty({n}, at::kBool, device);
    check(lib.ash_grid_query(map_of(handle), ptr<float>(x), n, grid_dim, ptr<int64_t>(grids),
                             ptr<int64_t>(cells), ptr<float>(offsets), ptr<uint8_t>(masks),
                             stream_of(device)));
    return {grids, cells, offsets, masks};
}

using Optional = std::optional<Tensor>;

// `t` on the device as contiguous float32
Tensor floats_on(const Tensor& t, int64_t device) {
    return t.to(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device)), at::kFloat).contiguous();
}

// ---------------------------------------------------------------------- rays
struct RayOperands {
    Tensor o, d, origin;
    RayOperands(const Tensor& origins, const Tensor& directions, const Optional& from, int64_t device) {
        o = floats_on(origins, device);
        d = floats_on(directions, device);
        need(o.dim() == 2 && o.size(1) == 3 && d.sizes() == o.sizes(),
             "ray origins and directions must both be (N, 3)");
        if (from.has_value()) origin = floats_on(*from, device);
    }
};

// Scratch of a call on rays for the map of the blocks in bounds (undefined: none), and
// what it is to be marked with.
struct Volume {
    Tensor bytes;
    int mark = 0;
    void* stream = nullptr;
    bool keep = false;
};

// The volumes that are kept for the next calls on rays, of any map, so that these need not
// clear theirs: up to eight of 4 MB, which go with the last map.  A volume is one call's
// alone from take to give, returns to calls on its own stream only, and what it holds
// of earlier calls is never looked at: every call marks its blocks with another number,
// and after the last the volume is cleared.  A captured call has one of its own, cleared by
// every replay.  (Near, far and samples of 32 768 rays, with one launch of two each less:
// 70 -> 62 us.)
class Volumes {
  public:
    // (held by every map)
    static std::shared_ptr<Volumes> shared() {
        static std::mutex mutex;
        static std::weak_ptr<Volumes> all;
        std::lock_guard<std::mutex> lock(mutex);
        auto those = all.lock();
        if (!those) all = those = std::make_shared<Volumes>();
        return those;
    }

    Volume take(const ash_map_t* map, int lo, int hi, int64_t n, int64_t samples, int64_t device) {
        Volume v;
        int64_t bytes = lib.ash_map_ray_volume_bytes(map, lo, hi, n, samples);
        if (bytes <= 0) return v;
        v.stream = stream_of(device);
        v.keep = lib.ash_ray_volume_kept(map, v.stream) != 0;
        if (!v.keep) bytes = lib.ash_ray_volume_bytes(lo, hi, n, samples != 0);
        if (bytes <= 0) return v;
        if (v.keep) {
            std::lock_guard<std::mutex> lock(mutex_);
            for (auto k = kept_.begin(); k != kept_.end(); ++k) {
                if (k->bytes.numel() != bytes || k->bytes.get_device() != device || k->stream != v.stream) continue;
                v = std::move(*k);
                kept_.erase(k);
                v.mark = v.mark < ASH_RAY_VOLUME_MARKS ? v.mark + 1 : 0;
                return v;
            }
        }
        v.bytes = empty({bytes}, at::kByte, device);
        return v;
    }

    // The launches that `v` was taken for are queued.
    void give(Volume&& v) {
        if (!v.keep) return;
        if (v.mark == 0) v.mark = 1;
        Tensor oldest;
        std::lock_guard<std::mutex> lock(mutex_);
        if (kept_.size() >= kMost) {
            oldest = std::move(kept_.front().bytes);
            kept_.erase(kept_.begin());
        }
        kept_.push_back(std::move(v));
    }

  private:
    static constexpr size_t kMost = 8;
    std::mutex mutex_;
    std::vector<Volume> kept_;
};

std::tuple<Tensor, Tensor> ray_near_far(uintptr_t handle, int64_t device, Volumes& volumes,
                                        const Tensor& origins,
                                        const Tensor& directions, const Optional& origin,
                                        double cell_size, const Tensor& bbox_min, const Tensor& bbox_max,
                                        double t_min, double t_max, double grid2cell, int block_lo,
                                        int block_hi) {
    const RayOperands r(origins, directions, origin, device);
    const Tensor lo = floats_on(bbox_min, device), hi = floats_on(bbox_max, device);
    need(lo.numel() == 3 && hi.numel() == 3, "the box has three coordinates per corner");
    const int64_t n = r.o.size(0);
    Tensor nears = empty({n}, at::kFloat, device), fars = empty({n}, at::kFloat, device);
    Volume volume = volumes.take(map_of(handle), block_lo, block_hi, n, 0, device);
    check(lib.ash_ray_find_near_far_marked(
            map_of(handle), ptr<uint8_t>(volume.bytes), block_lo, block_hi, volume.mark, ptr<float>(r.o),
            ptr<float>(r.d), ptr<float>(r.origin), static_cast<float>(cell_size), ptr<float>(lo),
            ptr<float>(hi), n, static_cast<float>(t_min), static_cast<float>(t_max),
            static_cast<float>(grid2cell), ptr<float>(nears), ptr<float>(fars), stream_of(device)));
    volumes.give(std::move(volume));
    return {nears, fars};
}

// A range per ray (world units, brought to cell units by the kernel), or one
// number for all of them, in world units as well.
struct RayRange {
    Tensor each;
    float for_all = 0.f;
    RayRange(const py::object& range, double cell_size, int64_t n, int64_t device) {
        if (THPVariable_Check(range.ptr())) {
            each = floats_on(py::cast<Tensor>(range), device).expand({n}).contiguous();
        } else {
            for_all = static_cast<float>(py::cast<double>(range) / cell_size);
        }
    }
};

// (ray_indices, t_nears, t_fars, prefix), or None where a ray has more samples
// than `stride`.
std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> ray_sample(
        uintptr_t handle, int64_t device, Volumes& volumes, const Tensor& origins, const Tensor& directions,
        const Optional& origin, double cell_size, const py::object& nears, const py::object& fars,
        int64_t max_samples, double grid2cell, int64_t stride, int block_lo, int block_hi) {
    const RayOperands r(origins, directions, origin, device);
    const int64_t n = r.o.size(0);
    const RayRange near(nears, cell_size, n, device), far(fars, cell_size, n, device);
    const Tensor counts = empty({n}, at::kLong, device), prefix = empty({n}, at::kLong, device);
    const Tensor groups = empty({lib.ash_ray_sample_groups(n), 2}, at::kLong, device);
    const Tensor stage = empty({n, stride, 2}, at::kFloat, device);
    Volume volume = volumes.take(map_of(handle), block_lo, block_hi, n, max_samples, device);
    void* stream = stream_of(device);
    int64_t out[2] = {0, 0};
    int status;
    {
        py::gil_scoped_release waits_for_the_device;
        status = lib.ash_ray_sample_march_marked(
                map_of(handle), ptr<uint8_t>(volume.bytes), block_lo, block_hi, volume.mark,
                ptr<float>(r.o), ptr<float>(r.d), ptr<float>(r.origin), static_cast<float>(cell_size), ptr<float>(near.each), ptr<float>(far.each),
                near.for_all, far.for_all, n, max_samples, static_cast<float>(grid2cell),
                ptr<int64_t>(counts), ptr<int64_t>(groups), ptr<float>(stage), stride, out, stream);
    }
    check(status);
    volumes.give(std::move(volume));
    if (out[1] > stride) return std::nullopt;
    Tensor indices = empty({out[0]}, at::kLong, device);
    Tensor t_nears = empty({out[0]}, at::kFloat, device), t_fars = empty({out[0]}, at::kFloat, device);
    check(lib.ash_ray_sample_place(ptr<int64_t>(counts), ptr<int64_t>(groups), ptr<float>(stage), stride,
                                   n, static_cast<float>(cell_size), ptr<int64_t>(indices),
                                   ptr<float>(t_nears), ptr<float>(t_fars), ptr<int64_t>(prefix), stream));
    return std::make_tuple(indices, t_nears, t_fars, prefix);
}

// (triangles, vertices).  `sdfs`, `weights`: a value per cell at the stride of
// their last dimension; `lut`, `grid_coords`, `grid_indices`: contiguous.
std::pair<Tensor, Tensor> surface_mesh(uintptr_t handle, int64_t device, const Tensor& sdfs,
                                       const Tensor& weights, const Tensor& grid_indices,
                                       const Tensor& grid_coords, const Tensor& lut, double iso,
                                       double weight_thr, bool to_world, double cell_to_world,
                                       const Optional& origin) {
    const int64_t b = sdfs.size(0), n = grid_indices.size(0);
    for (const Tensor* t : {&sdfs, &weights, &grid_indices, &grid_coords, &lut}) {
        need(t->is_cuda() && t->get_device() == device, "all tensors must be on the map's device");
    }
    for (const Tensor* t : {&sdfs, &weights}) {
        need(t->dim() == 2 && t->size(0) == b && t->size(1) == 512 && t->scalar_type() == sdfs.scalar_type() &&
                     (b == 1 || t->stride(0) == 512 * t->stride(1)),
             "field and weights must be (num_embeddings, 512), evenly strided, of one type");
    }
    need(sdfs.scalar_type() == at::kFloat || sdfs.scalar_type() == at::kDouble,
         "sdfs must be float32 or float64");
    need(grid_indices.scalar_type() == at::kLong && grid_indices.dim() == 1 &&
                 lut.scalar_type() == at::kLong && lut.dim() == 2 && lut.size(0) == b && lut.size(1) == 8 &&
                 grid_coords.scalar_type() == at::kInt && grid_coords.dim() == 2 &&
                 grid_coords.size(0) == b && grid_coords.size(1) == 3 && grid_indices.is_contiguous() &&
                 lut.is_contiguous() && grid_coords.is_contiguous(),
         "coordinate / neighbour tables do not match the grid");
    Tensor from;
    if (origin.has_value()) from = floats_on(*origin, device);
    const int32_t dtype = sdfs.scalar_type() == at::kFloat ? ASH_F32 : ASH_F64;
    const Tensor workspace = empty({lib.ash_surface_block8_workspace_bytes(n, b)}, at::kByte, device);
    void* stream = stream_of(device);
    int64_t out[2] = {0, 0};
    int status;
    {
        py::gil_scoped_release waits_for_the_device;
        status = lib.ash_surface_block8_classify(
                map_of(handle), ptr<void>(sdfs), sdfs.stride(1), ptr<void>(weights), weights.stride(1),
                ptr<int64_t>(grid_indices), ptr<int64_t>(lut), n, b, static_cast<float>(iso),
                static_cast<float>(weight_thr), dtype, ptr<void>(workspace), out, stream);
    }
    check(status);
    const Tensor vertices = empty({out[0], 3}, at::kFloat, device);
    const Tensor triangles = empty({out[1], 3}, at::kInt, device);
    check(lib.ash_surface_block8_extract(
            ptr<void>(sdfs), sdfs.stride(1), ptr<int64_t>(grid_indices), ptr<int32_t>(grid_coords),
            ptr<int64_t>(lut), n, b, static_cast<float>(iso), dtype, ptr<void>(workspace), out[0], out[1],
            to_world, static_cast<float>(cell_to_world), ptr<float>(from), ptr<float>(vertices),
            ptr<int32_t>(triangles), stream));
    return {triangles, vertices};
}

Tensor table_of(const Tensor& t, int64_t rows, int64_t device, const char* name) {
    if (!t.is_cuda() || t.get_device() != device || t.scalar_type() != at::kLong || t.dim() != 2 ||
        t.size(0) != rows || t.size(1) != 8) {
        fail(std::string(name) + " must be int64 (" + std::to_string(rows) + ", 8) on cuda:" +
             std::to_string(device));
    }
    return t.contiguous();
}

void fuse_frame(uintptr_t handle, int64_t device, const Tensor& positions_in, const Optional& origin,
                double cell_size, int dilation, bool bidirectional, int bound_lo, int bound_hi,
                const Tensor& touched, const Tensor& coords, const Tensor& emb, int grid_dim,
                double cell_to_world, const Optional& world_origin, const Tensor& intrinsic_in,
                const Tensor& extrinsic_in, const Tensor& depth_in, const Optional& color_in,
                double trunc, double depth_max, const Optional& counts) {
    const Tensor x = positions_of(positions_in);
    need(x.is_cuda() && x.get_device() == device, "positions must be on the map's device");
    need(emb.is_cuda() && emb.get_device() == device && emb.scalar_type() == at::kFloat &&
                 emb.is_contiguous(),
         "embeddings must be contiguous float32 on the map's device");
    need(emb.dim() == 3 && emb.size(1) == static_cast<int64_t>(grid_dim) * grid_dim * grid_dim,
         "embeddings must be (num_embeddings, grid_dim^3, embedding_dim)");
    need(emb.size(0) >= touched.size(0), "one embedding row per index of the map is needed");
    const Tensor intrinsic = floats_on(intrinsic_in, device), extrinsic = floats_on(extrinsic_in, device);
    need(intrinsic.dim() == 2 && intrinsic.size(0) == 3 && intrinsic.size(1) == 3 &&
                 extrinsic.dim() == 2 && extrinsic.size(0) == 4 && extrinsic.size(1) == 4,
         "intrinsic must be 3x3 and extrinsic 4x4");
    const Tensor depth = floats_on(depth_in, device);
    need(depth.dim() == 2, "depth must be (H, W)");
    Tensor color, from, to;
    if (color_in.has_value()) {
        color = floats_on(*color_in, device);
        need(color.dim() == 3 && color.size(0) == depth.size(0) && color.size(1) == depth.size(1) &&
                     color.size(2) == 3,
             "color must be (H, W, 3)");
    }
    if (origin.has_value()) from = floats_on(*origin, device);
    if (world_origin.has_value()) to = floats_on(*world_origin, device);
    ash_map_t* map = map_of(handle);
    void* stream = stream_of(device);
    int64_t scratch_bytes = 0;
    check(lib.ash_map_insert_scratch_bytes(map, 0, 0, nullptr, ASH_STREAMING_NEVER, &scratch_bytes));
    const Tensor scratch = scratch_bytes > 0 ? empty({scratch_bytes}, at::kByte, device) : Tensor();
    int status;
    {
        py::gil_scoped_release may_wait;
        status = lib.ash_map_upkeep(map, x.size(0), ptr<void>(scratch), scratch_bytes, nullptr, stream);
    }
    check(status);
    check(lib.ash_grid_fuse_frame(
            map, ptr<float>(x), x.size(0), ptr<float>(from), static_cast<float>(cell_size), dilation,
            bidirectional, bound_lo, bound_hi, ptr<uint8_t>(touched), ptr<int32_t>(coords),
            ptr<float>(emb), emb.size(0), grid_dim, static_cast<int>(emb.size(2)),
            static_cast<float>(cell_to_world), ptr<float>(to), ptr<float>(intrinsic),
            ptr<float>(extrinsic), ptr<float>(depth), ptr<float>(color),
            static_cast<int>(depth.size(0)), static_cast<int>(depth.size(1)),
            static_cast<float>(trunc), static_cast<float>(depth_max),
            counts.has_value() ? ptr<int32_t>(*counts) : nullptr, stream));
}

// (features, masks, grid_indices, cell_indices, offsets); the last three None
// unless `need_operands`.
std::tuple<Tensor, Tensor, Optional, Optional, Optional> grid_forward(
        uintptr_t handle, int64_t device, const Tensor& x_in, const Tensor& emb, const Tensor& lut_g,
        const Tensor& lut_c2c, const Tensor& lut_c2g, int grid_dim, const std::string& interpolation,
        bool need_operands, const Optional& origin_in, double cell_size) {
    ash_query_args args = {};
    args.interpolation = interpolation_of(interpolation);
    args.dtype = dtype_of(emb, "embeddings");
    need(emb.dim() == 3 && emb.is_contiguous(),
         "embeddings must be contiguous (num_embeddings, cells_per_grid, dim)");
    if (!emb.is_cuda()) fail("embeddings must live on a HIP device, got " + emb.device().str());
    if (emb.get_device() != device) {
        fail("the map is on cuda:" + std::to_string(device) + ", embeddings on " + emb.device().str());
    }
    need(x_in.dim() == 2 && x_in.size(1) == 3 && x_in.scalar_type() == at::kFloat && x_in.is_cuda() &&
                 x_in.get_device() == device,
         "positions must be float32 (N, 3) on the device of the embeddings");
    const Tensor x = x_in.contiguous();
    Tensor origin;
    if (origin_in.has_value()) {
        need(origin_in->is_cuda() && origin_in->get_device() == device &&
                     origin_in->scalar_type() == at::kFloat && origin_in->numel() == 3,
             "origin must be three float32 on the device of the embeddings");
        origin = origin_in->contiguous();
    }
    const int64_t b = emb.size(0), m = emb.size(1), e = emb.size(2), n = x.size(0);
    const Tensor g = table_of(lut_g, b, device, "lut_grid_nb2grid_idx");
    const Tensor c2c = table_of(lut_c2c, m, device, "lut_cell_nb2cell_idx");
    const Tensor c2g = table_of(lut_c2g, m, device, "lut_cell_nb2grid_nb");
    args.embeddings = emb.data_ptr();
    args.lut_grid_nb2grid_idx = ptr<int64_t>(g);
    args.lut_cell_nb2cell_idx = ptr<int64_t>(c2c);
    args.lut_cell_nb2grid_nb = ptr<int64_t>(c2g);
    args.num_queries = n;
    args.num_embeddings = b;
    args.cells_per_grid = m;
    args.embedding_dim = e;
    Tensor out = empty({n, e}, emb.scalar_type(), device), masks = empty({n}, at::kBool, device);
    Tensor grids, cells, offsets;
    if (need_operands) {
        grids = empty({n}, at::kLong, device);
        cells = empty({n}, at::kLong, device);
        offsets = empty({n, 3}, at::kFloat, device);
    }
    check(lib.ash_grid_forward(map_of(handle), ptr<float>(x), ptr<float>(origin),
                               static_cast<float>(cell_size), grid_dim, &args, out.data_ptr(),
                               ptr<uint8_t>(masks), ptr<int64_t>(grids), ptr<int64_t>(cells),
                               ptr<float>(offsets), stream_of(device)));
    if (!need_operands) return {out, masks, Optional(), Optional(), Optional()};
    return {out, masks, grids, cells, offsets};
}

// The operands of the three query functions: checked, contiguous, held while
// the launch is issued.
struct Operands {
    ash_query_args args = {};
    Tensor emb, held[7];
    int64_t device, n, e;

    Operands(const std::vector<Tensor>& in, const std::string& interpolation) {
        static const char* const names[] = {"offsets", "grid_indices", "cell_indices", "masks",
                                            "lut_grid_nb2grid_idx", "lut_cell_nb2cell_idx",
                                            "lut_cell_nb2grid_nb"};
        need(in.size() == 8, "a query takes the embeddings and seven operands");
        args.interpolation = interpolation_of(interpolation);
        args.dtype = dtype_of(in[0], "embeddings");
        need(in[0].dim() == 3, "embeddings must be (num_embeddings, cells_per_grid, dim)");
        if (!in[0].is_cuda()) fail("embeddings must live on a HIP device, got " + in[0].device().str());
        emb = in[0].contiguous();
        device = emb.get_device();
        n = in[2].dim() > 0 ? in[2].size(0) : 0;
        const int64_t b = emb.size(0), m = emb.size(1);
        e = emb.size(2);
        const int64_t numel[7] = {n * 3, n, n, n, b * 8, m * 8, m * 8};
        const at::ScalarType type[7] = {at::kFloat, at::kLong, at::kLong, at::kBool,
                                        at::kLong, at::kLong, at::kLong};
        for (int t = 0; t < 7; ++t) {
            const Tensor& x = in[t + 1];
            if (x.device() != emb.device()) {
                fail(std::string(names[t]) + " is on " + x.device().str() + ", embeddings on " +
                     emb.device().str());
            }
            if (x.scalar_type() != type[t]) {
                fail(std::string(names[t]) + " must be " + c10::toString(type[t]) + ", got " +
                     c10::toString(x.scalar_type()));
            }
            if (x.numel() != numel[t]) {
                fail(std::string(names[t]) + " has shape " + shape_of(x) + ", expected " +
                     std::to_string(numel[t]) + " elements");
            }
            held[t] = x.contiguous();
        }
        args.embeddings = emb.data_ptr();
        args.offsets = ptr<float>(held[0]);
        args.grid_indices = ptr<int64_t>(held[1]);
        args.cell_indices = ptr<int64_t>(held[2]);
        args.masks = ptr<uint8_t>(held[3]);
        args.lut_grid_nb2grid_idx = ptr<int64_t>(held[4]);
        args.lut_cell_nb2cell_idx = ptr<int64_t>(held[5]);
        args.lut_cell_nb2grid_nb = ptr<int64_t>(held[6]);
        args.num_queries = n;
        args.num_embeddings = b;
        args.cells_per_grid = m;
        args.embedding_dim = e;
    }

    // `t` has to be a tensor like the embeddings with n x width elements
    void must_be_like(const Tensor& t, int64_t width, const char* name) const {
        if (t.device() != emb.device()) {
            fail(std::string(name) + " is on " + t.device().str() + ", embeddings on " + emb.device().str());
        }
        if (t.scalar_type() != emb.scalar_type()) {
            fail(std::string(name) + " must be " + c10::toString(emb.scalar_type()) + ", got " +
                 c10::toString(t.scalar_type()));
        }
        if (t.numel() != n * width) {
            fail(std::string(name) + " has shape " + shape_of(t) + ", expected (" + std::to_string(n) +
                 ", " + std::to_string(width) + ")");
        }
    }

    Tensor like(const Tensor& t, int64_t width, const char* name) const {
        must_be_like(t, width, name);
        return t.contiguous();
    }

    // What a gradient with respect to offsets is multiplied by to be that with respect
    // to positions in units of a cell: torch, too, divides by a number by multiplying
    // with its reciprocal, rounded from float64 to the tensor's type.
    static double per_position(double cell_size) { return 1.0 / cell_size; }

    Tensor output(int64_t width) const { return empty({n, width}, emb.scalar_type(), device); }

    // where the embedding gradient goes: a new tensor, or `into` added to
    Tensor gradient(const Optional& into, bool wanted) const {
        if (!into.has_value()) return wanted ? at::empty_like(emb) : Tensor();
        need(into->sizes() == emb.sizes() && into->scalar_type() == emb.scalar_type() &&
                     into->device() == emb.device() && into->is_contiguous(),
             "accumulate_into must be a contiguous tensor like the embeddings");
        return *into;
    }
};

Optional maybe(const Tensor& t) { return t.defined() ? Optional(t) : Optional(); }

Tensor query_forward(const std::vector<Tensor>& operands, const std::string& interpolation) {
    Operands q(operands, interpolation);
    Tensor out = q.output(q.e);
    check(lib.ash_query_forward(&q.args, out.data_ptr(), stream_of(q.device)));
    return out;
}

std::tuple<Optional, Optional> query_backward_forward(const Tensor& z_in, const std::vector<Tensor>& operands,
                                                      const std::string& interpolation,
                                                      bool need_embeddings, bool need_offsets,
                                                      const Optional& accumulate_into, double cell_size) {
    Operands q(operands, interpolation);
    const Tensor z = q.like(z_in, q.e, "z");
    const Tensor grad = q.gradient(accumulate_into, need_embeddings);
    const Tensor offsets = need_offsets ? q.output(3) : Tensor();
    check(lib.ash_query_backward_forward_scaled(&q.args, z.data_ptr(), nullptr, nullptr, ptr<void>(grad),
                                                ptr<void>(offsets), q.per_position(cell_size),
                                                accumulate_into.has_value(), stream_of(q.device)));
    return {maybe(grad), maybe(offsets)};
}

std::tuple<Tensor, Optional> query_backward_both(const Tensor& z_in, const Tensor& gg_in,
                                                 const Tensor& z_second_in,
                                                 const std::vector<Tensor>& operands,
                                                 const std::string& interpolation, bool need_offsets,
                                                 const Optional& accumulate_into, double cell_size) {
    Operands q(operands, interpolation);
    const Tensor z = q.like(z_in, q.e, "z"), gg = q.like(gg_in, 3, "grad_grad_offsets");
    const Tensor z_second = q.like(z_second_in, q.e, "z of the second order");
    const Tensor grad = q.gradient(accumulate_into, true);
    const Tensor offsets = need_offsets ? q.output(3) : Tensor();
    check(lib.ash_query_backward_forward_scaled(
            &q.args, z.data_ptr(), gg.data_ptr(), z_second.data_ptr(), grad.data_ptr(), ptr<void>(offsets),
            q.per_position(cell_size), accumulate_into.has_value(), stream_of(q.device)));
    return {grad, maybe(offsets)};
}

std::tuple<Optional, Optional> query_backward_backward(const Tensor& gg_in, const Tensor& z_in,
                                                       const std::vector<Tensor>& operands,
                                                       const std::string& interpolation, bool need_z,
                                                       bool need_embeddings,
                                                       const Optional& accumulate_into, double cell_size) {
    Operands q(operands, interpolation);
    const Tensor z = q.like(z_in, q.e, "z"), gg = q.like(gg_in, 3, "grad_grad_offsets");
    const Tensor grad_z = need_z ? q.output(q.e) : Tensor();
    const Tensor grad = q.gradient(accumulate_into, need_embeddings);
    check(lib.ash_query_backward_backward_scaled(&q.args, gg.data_ptr(), z.data_ptr(), ptr<void>(grad_z),
                                                 ptr<void>(grad), q.per_position(cell_size),
                                                 accumulate_into.has_value(), stream_of(q.device)));
    return {maybe(grad_z), maybe(grad)};
}

// The embedding gradient of a query_backward_backward whose contributions are
// still to come (query_backward_both): `accumulate_into`, or zeros.  Everything is
// checked here, where the call is made, and made contiguous where it is read.
Tensor query_gradient_later(const Tensor& gg_in, const Tensor& z_in, const std::vector<Tensor>& operands,
                            const std::string& interpolation, const Optional& accumulate_into) {
    Operands q(operands, interpolation);
    q.must_be_like(z_in, q.e, "z");
    q.must_be_like(gg_in, 3, "grad_grad_offsets");
    const Tensor grad = q.gradient(accumulate_into, true);
    if (!accumulate_into.has_value()) {
        q.args.num_queries = 0;   // nothing but the zeros
        check(lib.ash_query_backward_forward(&q.args, nullptr, grad.data_ptr(), nullptr, stream_of(q.device)));
    }
    return grad;
}

// Whether nobody looks at the gradient that the node of `ctx` hands to the node
// behind its input `input`: no hook behind the one or before the other.
bool hands_over_unseen(const py::object& ctx, size_t input) {
    if (!THPFunction_Check(ctx.ptr())) return false;
    const auto node = reinterpret_cast<THPFunction*>(ctx.ptr())->cdata.lock();
    if (!node || input >= node->num_outputs() || !node->post_hooks().empty()) return false;
    const auto& next = node->next_edge(input).function;
    return next && next->pre_hooks().empty() && next->tensor_pre_hooks().empty() &&
           next->retains_grad_hooks().empty();
}

// Whether the running backward pass consumes the gradient that the node of `ctx`
// makes for its input `input` (`through`: the input belongs to a forward node's copy of
// a tensor, and the node asked about is the one behind that node's first input).  As
// torch._C._will_engine_execute_node says it of a Python object of the node, without
// the object, and without the exception it raises for a leaf whose gradient is what
// the pass was asked for (13 us of a training step); outside a pass: yes.
bool grad_requested(const py::object& ctx, size_t input, bool through) {
    if (!THPFunction_Check(ctx.ptr())) return true;
    const auto function = reinterpret_cast<THPFunction*>(ctx.ptr());
    const auto node = function->cdata.lock();
    if (!node || input >= node->num_outputs()) return true;
    const PyObject* wanted = PyTuple_GetItem(function->needs_input_grad, static_cast<Py_ssize_t>(input));
    if (wanted == nullptr) throw py::error_already_set();
    if (wanted != Py_True) return false;
    auto behind = node->next_edge(input).function;
    if (behind && through) {
        if (behind->num_outputs() == 0) return true;
        behind = behind->next_edge(0).function;
    }
    if (!behind) return false;
    const auto* executed = torch::autograd::get_current_graph_task_exec_info();
    const auto* all = torch::autograd::get_current_graph_task_nodes_in_graph();
    if (executed == nullptr || all == nullptr) return true;
    if (all->find(behind.get()) == all->end()) return false;
    if (executed->empty()) return true;
    const auto it = executed->find(behind.get());
    return it != executed->end() && it->second.should_execute();
}

std::tuple<Optional, Tensor, std::vector<Tensor>> find_rows_py(uintptr_t handle, int64_t dim, int64_t device,
                                                               const Tensor& keys,
                                                               const std::vector<Tensor>& tables,
                                                               bool zero_misses, bool need_indices) {
    auto [indices, masks, rows] = find_rows(handle, dim, device, keys, tables, zero_misses, need_indices);
    return {maybe(indices), masks, rows};
}

}  // namespace

PYBIND11_MODULE(_ash_host, m) {
    m.doc() = "host side of libash_hip.so's calls on torch tensors";
    // (build.py: host_fingerprint)
    m.attr("source_fingerprint") = ASH_HOST_FINGERPRINT;
    m.def("bind", &bind);
    m.def("find", &find);
    m.def("finds_rows_of", &finds_rows_of);
    m.def("find_rows", &find_rows_py);
    m.def("embedding_rows", &embedding_rows);
    m.def("gather_rows", &gather_rows);
    m.def("insert", &insert);
    m.def("erase", &erase);
    m.def("can_zero", &can_zero);
    m.def("clear", &clear);
    m.def("counters", &counters);
    m.def("items", &items);
    m.def("items_rows", &items_rows);
    m.def("neighbors", &neighbors);
    m.def("query_cells", &query_cells);
    m.def("grid_forward", &grid_forward);
    m.def("fuse_frame", &fuse_frame);
    py::class_<Volumes, std::shared_ptr<Volumes>>(m, "Volumes").def(py::init(&Volumes::shared));
    m.def("ray_near_far", &ray_near_far);
    m.def("ray_sample", &ray_sample);
    m.def("surface_mesh", &surface_mesh);
    m.def("query_forward", &query_forward);
    using py::arg;
    m.def("query_backward_forward", &query_backward_forward, arg("z"), arg("operands"), arg("interpolation"),
          arg("need_embeddings"), arg("need_offsets"), arg("accumulate_into"), arg("cell_size") = 1.0);
    m.def("query_backward_both", &query_backward_both, arg("z"), arg("grad_grad_offsets"), arg("z_second"),
          arg("operands"), arg("interpolation"), arg("need_offsets"), arg("accumulate_into"),
          arg("cell_size") = 1.0);
    m.def("query_gradient_later", &query_gradient_later);
    m.def("hands_over_unseen", &hands_over_unseen);
    m.def("grad_requested", &grad_requested);
    m.def("query_backward_backward", &query_backward_backward, arg("grad_grad_offsets"), arg("z"),
          arg("operands"), arg("interpolation"), arg("need_z"), arg("need_embeddings"),
          arg("accumulate_into"), arg("cell_size") = 1.0);
}

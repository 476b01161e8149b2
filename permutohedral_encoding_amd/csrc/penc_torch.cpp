// The path from PermutoEncoding.forward() to the kernels and back through autograd, in native code.
//
// What bounds a call on a small batch is not the kernels (4 us for a thousand points) but what the host does
// around them: argument checks, output and workspace allocation, stream look-up and foreign-function
// calls cost 20 us per call when they run in the interpreter, and every backward node written in Python
// has to take the interpreter lock on the autograd thread besides.  Here the module makes one call into
// this extension; the two differentiable steps are autograd nodes of their own (EncodeNode for the
// slicing, EncodeBackNode for its gradients, which makes them differentiable once more), so a backward pass never enters
// the interpreter.  The kernels are reached through the C ABI of include/penc.h, from the library the
// Python side has loaded (bind()).
//
// The nodes follow the pair of autograd functions in funcs.py (reference: src/pytorch_modules/funcs.py), with one
// difference in form: the result is the (N, F(L+E)) view the module hands out rather than the (L+E, F, N)
// array behind it (reference: src/pytorch_modules/modules.py:87), so that the permute and reshape need no nodes.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <Python.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/functions/accumulate_grad.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/object_ptr.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_set>
#include <utility>
#include <vector>

#include "../../include/penc.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::variable_list;

// ------------------------------------------------------------------------------------------
// the C ABI

struct Api {
#define PENC_FN(name) decltype(&penc_##name) name = nullptr
    PENC_FN(status_string);
    PENC_FN(extra_levels);
    PENC_FN(forward);
    PENC_FN(forward_half);
    PENC_FN(forward_rowmajor);
    PENC_FN(forward_rowmajor_workspace_bytes);
    PENC_FN(scatter_workspace_bytes);
    PENC_FN(scatter_useful_bytes);
    PENC_FN(positions_workspace_bytes);
    PENC_FN(backward);
    PENC_FN(backward_half);
    PENC_FN(backward_rowmajor);
    PENC_FN(backward_sparse);
    PENC_FN(backward_both_orders);
    PENC_FN(double_backward_from_positions);
    PENC_FN(double_backward_from_positions_half);
    PENC_FN(double_backward_from_positions_rowmajor);
    PENC_FN(double_backward_from_positions_sparse);
    PENC_FN(adamw_step);
    PENC_FN(adamw_step_sparse);
    PENC_FN(upload);
    PENC_FN(backward_positions_rowmajor);
    PENC_FN(grad_grad_rowmajor);
    PENC_FN(slopes_bytes);
    PENC_FN(forward_cells);
    PENC_FN(forward_cells_workspace_bytes);
    PENC_FN(table_cells);
    PENC_FN(table_cells_workspace_bytes);
    PENC_FN(forward_slopes);
    PENC_FN(backward_positions_slopes);
    PENC_FN(grad_grad_slopes);
#undef PENC_FN
} api;

void check(int status, const char* what) {
    if (status != PENC_OK) TORCH_CHECK(false, what, ": ", api.status_string(status), " (status ", status, ")");
}

#define PENC_REQUIRE(cond, ...) TORCH_CHECK_VALUE(cond, __VA_ARGS__)

void require_f32_gpu(const Tensor& t, const char* name, int64_t ndim) {
    PENC_REQUIRE(t.is_cuda(), name, " should be in GPU memory. Please call .cuda() on the tensor");
    PENC_REQUIRE(t.scalar_type() == at::kFloat, name, " should be of type float");
    PENC_REQUIRE(t.dim() == ndim, name, " should have ", ndim, " dimensions, however it has sizes ", t.sizes());
}

void* current_stream(const at::Device& device) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream();
}

// The capture that a stream takes part in, 0 where it takes part in none.
uint64_t capture_of(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) {  // (the default stream while another is captured)
        (void)hipGetLastError();
        return 0;
    }
    return status == hipStreamCaptureStatusNone ? 0 : id + 1;
}

const float* data(const Tensor& t) { return static_cast<const float*>(t.const_data_ptr()); }
float* mutable_data(const Tensor& t) { return t.defined() ? static_cast<float*>(t.mutable_data_ptr()) : nullptr; }

// ------------------------------------------------------------------------------------------
// what one call of the encoding and its derivatives share

// A reference to a Python object that native code may drop from any thread.
struct PyRef {
    explicit PyRef(PyObject* o) : object(o) { Py_XINCREF(object); }
    PyRef(const PyRef&) = delete;
    PyRef& operator=(const PyRef&) = delete;
    ~PyRef() {
        if (object == nullptr || !Py_IsInitialized()) return;
        const PyGILState_STATE gil = PyGILState_Ensure();
        Py_DECREF(object);
        PyGILState_Release(gil);
    }
    PyObject* object;
};

struct Call {
    int pos_dim, feat, levels, capacity, extra, concat;
    float scaling;
    int table_format;  // 0: fp32, else PENC_TABLE_FP16 / PENC_TABLE_BF16, with PENC_TABLE_CELLS where in_cells
    bool in_cells;     // the table is a 16-bit copy in cells (table_in_cells)
    bool rows_output;
    int64_t n, levels_per_pass, max_workspace;  // the binding's LEVELS_PER_PASS, MAX_WORKSPACE_BYTES (< 0: no cap)
    Tensor positions;                           // contiguous
    Tensor table;                               // what the kernels gather from: the parameter or its 16-bit copy
    Tensor lattice_values;                      // the parameter
    Tensor scale_factor, shift, window;
    std::shared_ptr<PyRef> sparse_owner;  // the wrapper that keeps the sparse table gradient; null: dense gradients
    bool want_table, want_positions;
    bool hooked = false;  // hooks are set on what a graph saves (looked at where slopes could be kept)

    int64_t columns() const { return static_cast<int64_t>(feat) * (levels + extra); }
    at::Device device() const { return positions.device(); }
};

// An (N, F(L+E)) array in [L+E][F][N] order: the result of the slicing, and the gradient w.r.t. an upstream gradient.
Tensor level_major_array(const Call& c) {
    return at::empty_strided({c.n, c.columns()}, {1, c.n}, c.positions.options().dtype(at::kFloat));
}

Tensor bytes(const Call& c, size_t n) { return at::empty({static_cast<int64_t>(n)}, c.positions.options().dtype(at::kByte)); }

// The sparse table gradient of the call's wrapper (created there by the first gradient call): gradient and map.
std::pair<Tensor, Tensor> sparse_gradient(const Call& c) {
    const PyGILState_STATE gil = PyGILState_Ensure();
    Tensor grad, touched;
    PyObject* const lv = THPVariable_Wrap(c.lattice_values);
    PyObject* const sparse = PyObject_CallMethod(c.sparse_owner->object, "sparse_grad_for", "O", lv);
    if (sparse != nullptr) {
        PyObject* const g = PyObject_GetAttrString(sparse, "grad");
        PyObject* const t = PyObject_GetAttrString(sparse, "touched");
        if (g != nullptr && t != nullptr && THPVariable_Check(g) && THPVariable_Check(t)) {
            grad = THPVariable_Unpack(g);
            touched = THPVariable_Unpack(t);
        }
        Py_XDECREF(g);
        Py_XDECREF(t);
        Py_DECREF(sparse);
    }
    Py_XDECREF(lv);
    if (PyErr_Occurred()) {
        python_error error;  // (such as the allocator's, as the interpreter would raise it)
        error.persist();
        PyGILState_Release(gil);
        throw error;
    }
    PyGILState_Release(gil);
    TORCH_CHECK(grad.defined() && touched.defined(), "the sparse table gradient could not be created");
    return {grad, touched};
}

// The upstream gradient as the kernels take it: rows of `row_stride` floats, or (row_stride == 0) the [L+E][F][N] array.
struct Upstream {
    Tensor values;
    int64_t row_stride = 0;
};

Upstream upstream_of(const Call& c, const Tensor& grad) {
    require_f32_gpu(grad, "grad_sliced_values_monolithic", 2);
    PENC_REQUIRE(grad.size(0) == c.n && grad.size(1) == c.columns(),
                 "grad_sliced_values_monolithic should be nr_resolutions x val_dim x nr_positions");
    PENC_REQUIRE(grad.device() == c.device(), "grad_sliced_values_monolithic must be on the same device as positions");
    const int64_t s_point = grad.stride(0), s_col = grad.stride(1);
    if (s_point == 1 && s_col == c.n) return {grad, 0};
    const auto rows = [&](const Tensor& t) {
        const int64_t s = t.stride(0);
        return t.stride(1) == 1 && s >= c.columns() && s % 2 == 0 && (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 7u) == 0 &&
               s * c.n < (int64_t{1} << 31);
    };
    if (rows(grad)) return {grad, s_point};
    const Tensor dense = grad.contiguous();  // any other layout: rows are what it is brought into (a streaming copy)
    if (rows(dense)) return {dense, dense.stride(0)};
    Tensor level_major = level_major_array(c);
    level_major.copy_(dense);
    return {level_major, 0};
}

// Memory of `size` bytes that a call does better with and can do without: whether `take`, which allocates it, has found it.  A request in vain makes
// the allocator release all it has cached, for the driver to be asked again by whatever follows; so once a device has refused, as much is not
// asked for again until the process could have a sixteenth of it more than then.  Slopes are not given back for it.
bool take_optional(const at::Device& device, int64_t size, const std::function<void()>& take);
Tensor optional_bytes(const Call& c, int64_t n) {
    Tensor t;
    take_optional(c.device(), n, [&] { t = bytes(c, static_cast<size_t>(n)); });
    return t;
}

// Scratch memory of one gradient call, undefined when the library would not use any.  The scatter counts every
// pair of features as a level.  `copy_bytes`: the level-major copy of a row-major upstream gradient, which the call
// cannot do without.  A request over the cap, or one the allocator cannot serve, is made again for fewer levels per
// pass and in the end without the scatter's part (the library then adds directly), as in _native.scatter_workspace, which does not ask for `extra`.
Tensor gradient_workspace(const Call& c, bool table, bool positions, int64_t copy_bytes) {
    if (c.levels_per_pass < 0 && copy_bytes == 0) return {};
    int64_t pos_bytes = positions ? static_cast<int64_t>(api.positions_workspace_bytes(c.pos_dim, c.n, c.levels)) : 0;
    const int64_t pair_levels = static_cast<int64_t>(c.levels) * (c.feat / 2);
    int64_t per_pass = c.levels_per_pass <= 0 ? pair_levels : std::min(c.levels_per_pass, pair_levels);
    if (!table || c.levels_per_pass < 0) per_pass = 0;
    // (asked for once, with all levels in a pass: what a dense gradient uses besides, lists of late adds or the slack of narrower bins)
    int64_t extra = per_pass == pair_levels && c.sparse_owner == nullptr
                        ? static_cast<int64_t>(api.scatter_useful_bytes(c.pos_dim, c.feat, c.n, c.levels, c.capacity))
                        : 0;
    while (true) {
        int64_t want = per_pass > 0 ? static_cast<int64_t>(api.scatter_workspace_bytes(c.pos_dim, c.n, static_cast<int>(pair_levels),
                                                                                      c.capacity, static_cast<int>(per_pass)))
                                    : 0;
        want = std::max(want, pos_bytes) + copy_bytes + extra;
        if (c.max_workspace < 0 || want <= c.max_workspace) {
            if (want == 0) return {};
            if (extra > 0) {
                const Tensor ws = optional_bytes(c, want);
                if (ws.defined()) return ws;
            } else {
                try {
                    return bytes(c, static_cast<size_t>(want));
                } catch (const c10::OutOfMemoryError&) {
                }
            }
        }
        if (extra > 0) {
            extra = 0;
        } else if (per_pass > 1) {
            per_pass /= 2;
        } else if (per_pass == 1 || pos_bytes > 0) {
            per_pass = pos_bytes = 0;
        } else if (copy_bytes > 0) {
            return bytes(c, static_cast<size_t>(copy_bytes));  // throws if even that fails
        } else {
            return {};
        }
    }
}

void* workspace_of(const Tensor& ws) { return ws.defined() ? ws.mutable_data_ptr() : nullptr; }
size_t workspace_size(const Tensor& ws) { return ws.defined() ? static_cast<size_t>(ws.numel()) : 0; }

// The version a tensor must still be at when a node that did not save the tensor itself runs.
struct ExpectedVersion {
    c10::VariableVersion counter;
    uint32_t expected = 0;
    bool set = false;

    void expect(const Tensor& t) {
        TORCH_CHECK(!t.is_inference(), "Inference tensors cannot be saved for backward: make a clone outside of inference mode");
        counter = torch::autograd::impl::version_counter(t);
        expected = counter.current_version();
        set = true;
    }
    bool holds() const { return !set || counter.current_version() == expected; }
    void check(const char* what) const {
        TORCH_CHECK(holds(),
                    "one of the variables needed for gradient computation has been modified by an inplace operation: ", what, " is at version ",
                    counter.current_version(), "; expected version ", expected, " instead");
    }
};

// The slopes of the encoded features (penc_forward_slopes), kept from the forward to the passes that differentiate w.r.t. the positions,
// as autograd keeps the tensors a node saves: freed with the graph.  What they were computed from must still be what a gathering kernel
// would read then; where it is not (a table stepped between forward and backward, a pass on another stream), that kernel runs.
// (A write that the version counter does not see, such as one through `.data`, is not noticed: modules.py says what to do after one.)
// A forward that nothing differentiates w.r.t. the positions in the end has written them for nothing (penc_slopes.hpp has the times).
// Nobody pays for them with an allocation that fails: a forward takes its result first and does without slopes where they do not fit, all
// that are alive on a device take at most a sixteenth of the memory the process may use there, and they are given back when that
// memory runs short (GiveBackSlopes).
struct Slopes {
    static constexpr int kMaxDevices = 64;
    static std::atomic<int64_t> held[kMaxDevices];

    // What an input must still be: unchanged in place, and not given other memory (`lattice_values.data = ...`), which is no change in place.
    struct Input {
        ExpectedVersion version;
        c10::Storage storage;  // (kept, so that no other memory can take its place)
        int64_t offset = 0;

        void expect(const Tensor& t) {
            version.expect(t);
            storage = t.storage();
            offset = t.storage_offset();
        }
        bool holds(const Tensor& t) const {
            return version.holds() && t.storage().unsafeGetStorageImpl() == storage.unsafeGetStorageImpl() && t.storage_offset() == offset;
        }
    } inputs[5];
    static std::array<const Tensor*, 5> inputs_of(const Call& c) { return {&c.table, &c.positions, &c.window, &c.shift, &c.scale_factor}; }
    void* stream;
    int device = -1;
    int64_t reserved = 0;  // counted in held[device]

    Slopes() = default;
    Slopes(const Slopes&) = delete;
    Slopes& operator=(const Slopes&) = delete;
    ~Slopes() {
        {
            std::lock_guard<std::mutex> lock(mutex);
            alive.erase(this);
        }
        if (reserved != 0) held[device] -= reserved;
    }
    // The slopes, or an undefined tensor where they do not stand for what a gathering kernel would read, or have been given back.
    Tensor usable(const Call& c) const {
        if (current_stream(c.device()) != stream) return {};
        const auto from = inputs_of(c);
        for (size_t i = 0; i < from.size(); ++i)
            if (!inputs[i].holds(*from[i])) return {};
        std::lock_guard<std::mutex> lock(mutex);
        return values;
    }
    // For the forward that has just filled them.
    void keep(Tensor filled) {
        std::lock_guard<std::mutex> lock(mutex);
        values = std::move(filled);
        alive.insert(this);
    }

    // What this process may use of a device's memory, and what of that is still to be had from the driver.
    static int64_t most_memory(int device) {
        return static_cast<int64_t>(static_cast<double>(at::cuda::getDeviceProperties(device)->totalGlobalMem) *
                                    c10::hip::HIPCachingAllocator::getMemoryFraction(static_cast<c10::DeviceIndex>(device)));
    }
    static int64_t memory_left(int device) {  // (of the current device)
        size_t free = 0, total = 0;
        {
            c10::hip::HIPStreamCaptureModeGuard in_a_capture_too{hipStreamCaptureModeRelaxed};
            C10_HIP_CHECK(hipMemGetInfo(&free, &total));
        }
        const auto stats = c10::hip::HIPCachingAllocator::getDeviceStats(static_cast<c10::DeviceIndex>(device));
        const int64_t taken = stats.reserved_bytes[static_cast<size_t>(c10::CachingAllocator::StatType::AGGREGATE)].current;
        return std::min(static_cast<int64_t>(free), most_memory(device) - taken);
    }

    // Whether hooks are on what a graph saves, such as those of checkpointing, which trade memory for a second computation: nothing
    // beside what they see is kept then.  With the GIL held: looking copies Python objects.
    static bool hooks_are_set() { return at::SavedTensorDefaultHooks::get_hooks().has_value(); }

    // For the forward that is about to run: null where none are kept.
    static std::shared_ptr<Slopes> make(const Call& c) {
        if (!c.want_positions || c.hooked || c.columns() > 255 || c.levels_per_pass < 0) return nullptr;
        const int64_t want = static_cast<int64_t>(api.slopes_bytes(c.pos_dim, c.feat, c.n, c.levels, c.capacity, c.table_format));
        if (want == 0 || (c.max_workspace >= 0 && want > c.max_workspace)) return nullptr;
        const auto from = inputs_of(c);
        for (const Tensor* t : from)
            if (t->is_inference()) return nullptr;
        const int device = c.device().index();
        if (device < 0 || device >= kMaxDevices) return nullptr;
        const int64_t most = most_memory(device) / 16;
        if (held[device].fetch_add(want) + want > most) {
            held[device] -= want;
            return nullptr;
        }
        auto slopes = std::make_shared<Slopes>();
        slopes->device = device;
        slopes->reserved = want;
        slopes->stream = current_stream(c.device());
        for (size_t i = 0; i < from.size(); ++i) slopes->inputs[i].expect(*from[i]);
        return slopes;
    }

    // Gives back the slopes of a device that no running pass reads.  The memory itself is freed after the lock has been left: a thread that
    // holds the lock must not wait for the allocator's, which the caller of GiveBackSlopes holds.
    static bool give_back(int device) {
        std::vector<Tensor> freed;
        {
            std::lock_guard<std::mutex> lock(mutex);
            for (auto it = alive.begin(); it != alive.end();) {
                Slopes* const s = *it;
                if (s->device != device) {
                    ++it;
                    continue;
                }
                freed.push_back(std::move(s->values));
                s->values = Tensor();
                held[device] -= s->reserved;
                s->reserved = 0;
                it = alive.erase(it);
            }
        }
        return !freed.empty();
    }

private:
    static std::mutex mutex;                    // of `values` and `alive`; nothing is allocated or freed on a device under it
    static std::unordered_set<Slopes*>& alive;  // those with values (never destroyed: a node may outlive the statics of this file)
    Tensor values;
};
std::atomic<int64_t> Slopes::held[Slopes::kMaxDevices] = {};
std::mutex Slopes::mutex;
std::unordered_set<Slopes*>& Slopes::alive = *new std::unordered_set<Slopes*>();

// What the caching allocator asks for memory, on the thread that allocates and with that device current, before it turns to the driver.  It
// does not say how much it needs: slopes are given back as soon as the driver has less than a quarter of the process's memory left, so that
// any smaller request finds what it would find without them.  (Once a program's blocks are all cached the allocator does not come here.)
class GiveBackSlopes : public c10::FreeMemoryCallback {
public:
    static thread_local bool not_for_this;  // the thread asks for memory that it can do without
    bool Execute() override {
        if (not_for_this) return false;
        try {
            const int device = c10::hip::current_device();
            if (device < 0 || device >= Slopes::kMaxDevices || Slopes::held[device] == 0) return false;
            if (Slopes::memory_left(device) >= Slopes::most_memory(device) / 4) return false;
            return Slopes::give_back(device);
        } catch (const std::exception&) {
            return false;  // (the allocation goes on as it would)
        }
    }
};
thread_local bool GiveBackSlopes::not_for_this = false;

bool take_optional(const at::Device& device, int64_t size, const std::function<void()>& take) {
    struct Refusal {
        std::mutex mutex;
        int64_t size = 0, available = 0;  // the last request in vain (0: none since one as large was served), and what there was to be had after it
    };
    static Refusal refusals[Slopes::kMaxDevices];
    const int index = device.index();
    if (index < 0 || index >= Slopes::kMaxDevices) return false;
    Refusal& last = refusals[index];
    // what the allocator has cached and what the driver still has for this process
    const auto available = [&] {
        const auto stats = c10::hip::HIPCachingAllocator::getDeviceStats(static_cast<c10::DeviceIndex>(index));
        constexpr auto kAll = static_cast<size_t>(c10::CachingAllocator::StatType::AGGREGATE);
        return Slopes::memory_left(index) + stats.reserved_bytes[kAll].current - stats.allocated_bytes[kAll].current;
    };
    int64_t wanted = 0;
    {
        std::lock_guard<std::mutex> lock(last.mutex);
        if (last.size != 0 && size >= last.size) wanted = last.available + size / 16;
    }
    if (wanted != 0 && available() < wanted) return false;
    struct Asking {
        Asking() { GiveBackSlopes::not_for_this = true; }
        ~Asking() { GiveBackSlopes::not_for_this = false; }
    };
    try {
        const Asking asking;
        take();
    } catch (const c10::OutOfMemoryError&) {
        const int64_t left = available();
        std::lock_guard<std::mutex> lock(last.mutex);
        last.size = size;
        last.available = left;
        return false;
    }
    if (wanted != 0) {
        std::lock_guard<std::mutex> lock(last.mutex);
        last.size = 0;
    }
    return true;
}

// ------------------------------------------------------------------------------------------
// the three computations (reference: Encoding<D,F>::forward, ::backward, ::double_backward_from_positions, src/Encoding.cu:55-334)

// Whether forward_in_cells is worth a call: small batches, far below where it pays, wait for the host.
bool may_go_by_cells(const Call& c) { return c.table_format == 0 && c.n * c.levels >= (int64_t{1} << 20); }

// The forward by way of a copy of the table in cells, where that pays and there is memory for it; false: not done.  `rows` is undefined where
// the result is `level_major`, which else is scratch and may be undefined; `slopes` where none are kept.
bool forward_in_cells(const Call& c, Tensor level_major, const Tensor& rows, const Tensor& slopes) {
    const size_t n = api.forward_cells_workspace_bytes(c.pos_dim, c.feat, c.n, c.levels, c.capacity, rows.defined() ? static_cast<int>(c.columns()) : 0);
    if (n == 0 || (c.max_workspace >= 0 && static_cast<int64_t>(n) > c.max_workspace)) return false;
    if (!level_major.defined()) level_major = level_major_array(c);  // (a forward in rows needs as much either way)
    const Tensor ws = optional_bytes(c, static_cast<int64_t>(n));
    if (!ws.defined()) return false;
    check(api.forward_cells(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table), data(c.scale_factor), data(c.shift),
                            data(c.window), mutable_data(level_major), mutable_data(rows), c.columns(), mutable_data(slopes), c.concat, c.scaling,
                            ws.mutable_data_ptr(), n, current_stream(c.device())),
          "forward_cells");
    return true;
}

// With `slopes` the forward leaves them behind; where their memory is refused, it is reset and the forward is the one without.
Tensor compute_forward(const Call& c, std::shared_ptr<Slopes>& slopes) {
    void* const stream = current_stream(c.device());
    const bool as_rows = c.rows_output && c.table_format == 0 && c.columns() <= 255;
    Tensor out = as_rows ? at::empty({c.n, c.columns()}, c.positions.options()) : level_major_array(c);
    if (slopes != nullptr) {
        Tensor level_major = out, kept;
        try {
            if (as_rows) level_major = level_major_array(c);
            kept = at::empty({slopes->reserved / 4}, c.positions.options().dtype(at::kFloat));
        } catch (const c10::OutOfMemoryError&) {
            slopes.reset();
        }
        if (slopes != nullptr) {
            if (!may_go_by_cells(c) || !forward_in_cells(c, level_major, as_rows ? out : Tensor(), kept))
                check(api.forward_slopes(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), c.table.const_data_ptr(), c.table_format,
                                         data(c.scale_factor), data(c.shift), data(c.window), mutable_data(level_major),
                                         as_rows ? mutable_data(out) : nullptr, c.columns(), mutable_data(kept), c.concat, c.scaling, stream),
                      "forward_slopes");
            slopes->keep(std::move(kept));
            return out;
        }
    }
    if (may_go_by_cells(c) && (as_rows ? forward_in_cells(c, {}, out, {}) : forward_in_cells(c, out, {}, {}))) return out;
    if (as_rows) {
        const Tensor ws = bytes(c, api.forward_rowmajor_workspace_bytes(c.pos_dim, c.feat, c.n, c.levels, c.concat));
        check(api.forward_rowmajor(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table), data(c.scale_factor),
                                   data(c.shift), data(c.window), mutable_data(out), c.columns(), c.concat, c.scaling,
                                   workspace_of(ws), workspace_size(ws), stream),
              "forward_rowmajor");
        return out;
    }
    if (c.table_format != 0)
        check(api.forward_half(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), c.table.const_data_ptr(), c.table_format,
                               data(c.scale_factor), data(c.shift), data(c.window), mutable_data(out), c.concat, c.scaling, stream),
              "forward");
    else
        check(api.forward(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table), data(c.scale_factor),
                          data(c.shift), data(c.window), mutable_data(out), c.concat, c.scaling, stream),
              "forward");
    return out;
}

struct Gradients {
    Tensor table, positions;  // undefined: not wanted (or, for the table, added into the sparse gradient)
};

// The table gradient that comes through a position gradient, handed on by the node that met it (see EncodeNode).
struct SecondOrderTerm {
    int task = -1;                  // the graph task it belongs to
    Tensor double_positions_grad;   // contiguous
    Upstream upstream;              // level-major
};

Gradients compute_backward(const Call& c, const Upstream& up, bool want_table, bool want_positions, const SecondOrderTerm* second = nullptr) {
    Gradients g;
    if (!want_table && !want_positions) return g;
    void* const stream = current_stream(c.device());
    const bool sparse = want_table && c.sparse_owner != nullptr;
    PENC_REQUIRE(!sparse || c.table_format == 0, "sparse_table_grad needs an fp32 table");
    if (want_positions) g.positions = at::empty({c.n, c.pos_dim}, c.positions.options());
    if (want_table && !sparse) g.table = at::empty(c.lattice_values.sizes(), c.positions.options());
    const bool rows = up.row_stride != 0;
    const int64_t copy_bytes = rows && want_positions ? 4 * static_cast<int64_t>(c.feat) * c.levels * c.n + 512 : 0;
    const Tensor ws = gradient_workspace(c, want_table, want_positions, copy_bytes);
    float* const tg = mutable_data(g.table);
    float* const pg = mutable_data(g.positions);
    if (want_table && second != nullptr) {
        std::pair<Tensor, Tensor> kept;
        if (sparse) kept = sparse_gradient(c);
        check(api.backward_both_orders(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), c.table.const_data_ptr(),
                                       c.table_format, data(c.scale_factor), data(c.shift), data(c.window), data(up.values), up.row_stride,
                                       data(second->double_positions_grad), data(second->upstream.values),
                                       sparse ? mutable_data(kept.first) : tg,
                                       sparse ? static_cast<uint32_t*>(kept.second.mutable_data_ptr()) : nullptr, pg, workspace_of(ws),
                                       workspace_size(ws), stream),
              "backward_both_orders");
    } else if (sparse) {
        const auto [grad, touched] = sparse_gradient(c);
        check(api.backward_sparse(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table), data(c.scale_factor),
                                  data(c.shift), data(c.window), data(up.values), up.row_stride, mutable_data(grad),
                                  static_cast<uint32_t*>(touched.mutable_data_ptr()), pg, workspace_of(ws), workspace_size(ws), stream),
              "backward_sparse");
    } else if (c.table_format != 0) {
        check(api.backward_half(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), c.table.const_data_ptr(), c.table_format,
                                data(c.scale_factor), data(c.shift), data(c.window), data(up.values), up.row_stride, tg, pg,
                                workspace_of(ws), workspace_size(ws), stream),
              "backward");
    } else if (rows) {
        check(api.backward_rowmajor(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table), data(c.scale_factor),
                                    data(c.shift), data(c.window), data(up.values), up.row_stride, tg, pg, workspace_of(ws),
                                    workspace_size(ws), stream),
              "backward");
    } else {
        check(api.backward(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table), data(c.scale_factor),
                           data(c.shift), data(c.window), data(up.values), tg, pg, workspace_of(ws), workspace_size(ws), stream),
              "backward");
    }
    return g;
}

Tensor checked_double_positions_grad(const Call& c, const Tensor& double_positions_grad) {
    require_f32_gpu(double_positions_grad, "double_positions_grad", 2);
    PENC_REQUIRE(double_positions_grad.size(0) == c.n && double_positions_grad.size(1) == c.pos_dim,
                 "double_positions_grad should be nr_positions x pos_dim");
    return double_positions_grad.detach().contiguous();
}

// The position gradient alone, from the slopes where the forward has kept them.  With `keep_copy`, of rows the level-major copy outlives
// the call and takes their place: a scatter that follows, and the double backward's, reads it coalesced, where rows cost it a sixth
// of its time.
Tensor compute_positions_backward(const Call& c, Upstream& up, const Tensor& slopes, bool keep_copy) {
    Tensor positions = at::empty({c.n, c.pos_dim}, c.positions.options());
    void* const stream = current_stream(c.device());
    Tensor level_major;
    if (up.row_stride != 0 && keep_copy) level_major = level_major_array(c);
    if (slopes.defined()) {
        check(api.backward_positions_slopes(c.pos_dim, c.feat, c.n, c.levels, data(slopes), data(c.window), data(up.values), up.row_stride,
                                            mutable_data(level_major), mutable_data(positions), stream),
              "backward_positions_slopes");
    } else {
        const Tensor ws = gradient_workspace(c, false, true, 0);
        check(api.backward_positions_rowmajor(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), c.table.const_data_ptr(),
                                              c.table_format, data(c.scale_factor), data(c.shift), data(c.window), data(up.values),
                                              up.row_stride, mutable_data(level_major), mutable_data(positions), workspace_of(ws),
                                              workspace_size(ws), stream),
              "backward_positions");
    }
    if (!level_major.defined()) return positions;
    // (the columns of concatenated points carry no gradient and are not read, but whoever saves the copy sees the whole of it)
    const int64_t encoded = static_cast<int64_t>(c.feat) * c.levels;
    if (c.extra != 0) level_major.narrow(1, encoded, c.columns() - encoded).copy_(up.values.narrow(1, encoded, c.columns() - encoded));
    up = {level_major, 0};
    return positions;
}

// The gradient w.r.t. an upstream gradient, as dense rows or in [L+E][F][N] order, from the slopes.
Tensor compute_grad_grad(const Call& c, const Tensor& slopes, const Tensor& double_positions_grad, bool as_rows) {
    Tensor out = as_rows ? at::empty({c.n, c.columns()}, c.positions.options()) : level_major_array(c);
    check(api.grad_grad_slopes(c.pos_dim, c.feat, c.n, c.levels, data(slopes), data(c.window), data(double_positions_grad), mutable_data(out),
                               as_rows ? c.columns() : 0, c.concat, current_stream(c.device())),
          "grad_grad_slopes");
    return out;
}

// The same as dense rows, gathered.
Tensor compute_grad_grad_rows(const Call& c, const Tensor& double_positions_grad) {
    Tensor rows = at::empty({c.n, c.columns()}, c.positions.options());
    const Tensor ws = bytes(c, api.forward_rowmajor_workspace_bytes(c.pos_dim, c.feat, c.n, c.levels, c.concat));
    check(api.grad_grad_rowmajor(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), c.table.const_data_ptr(), c.table_format,
                                 data(c.scale_factor), data(c.shift), data(c.window), data(double_positions_grad), mutable_data(rows),
                                 c.columns(), c.concat, workspace_of(ws), workspace_size(ws), current_stream(c.device())),
          "grad_grad");
    return rows;
}

struct SecondOrder {
    Tensor table, upstream;  // gradients w.r.t. the table (undefined as above) and w.r.t. the upstream gradient
};

SecondOrder compute_double_backward(const Call& c, const Tensor& double_positions_grad, const Upstream& up, bool want_table,
                                    bool want_upstream) {
    const Tensor dpos = checked_double_positions_grad(c, double_positions_grad);
    void* const stream = current_stream(c.device());
    SecondOrder s;
    if (want_upstream) s.upstream = level_major_array(c);
    const bool sparse = want_table && c.sparse_owner != nullptr;
    if (want_table && !sparse) s.table = at::empty(c.lattice_values.sizes(), c.positions.options());
    const Tensor ws = want_table ? gradient_workspace(c, true, false, 0) : Tensor();
    float* const tg = mutable_data(s.table);
    float* const gg = mutable_data(s.upstream);
    if (sparse) {
        PENC_REQUIRE(c.table_format == 0, "sparse_table_grad needs an fp32 table");
        const auto [grad, touched] = sparse_gradient(c);
        check(api.double_backward_from_positions_sparse(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table),
                                                        data(c.scale_factor), data(c.shift), data(c.window), data(dpos), data(up.values),
                                                        up.row_stride, mutable_data(grad),
                                                        static_cast<uint32_t*>(touched.mutable_data_ptr()), gg, c.concat,
                                                        workspace_of(ws), workspace_size(ws), stream),
              "double_backward_from_positions_sparse");
    } else if (c.table_format != 0) {
        check(api.double_backward_from_positions_half(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions),
                                                      c.table.const_data_ptr(), c.table_format, data(c.scale_factor), data(c.shift),
                                                      data(c.window), data(dpos), data(up.values), up.row_stride, tg, gg, c.concat,
                                                      workspace_of(ws), workspace_size(ws), stream),
              "double_backward_from_positions");
    } else if (up.row_stride != 0) {
        check(api.double_backward_from_positions_rowmajor(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table),
                                                          data(c.scale_factor), data(c.shift), data(c.window), data(dpos),
                                                          data(up.values), up.row_stride, tg, gg, c.concat, workspace_of(ws),
                                                          workspace_size(ws), stream),
              "double_backward_from_positions");
    } else {
        check(api.double_backward_from_positions(c.pos_dim, c.feat, c.n, c.levels, c.capacity, data(c.positions), data(c.table),
                                                 data(c.scale_factor), data(c.shift), data(c.window), data(dpos), data(up.values), tg, gg,
                                                 c.concat, workspace_of(ws), workspace_size(ws), stream),
              "double_backward_from_positions");
    }
    return s;
}

// ------------------------------------------------------------------------------------------
// autograd

// The nodes compute through raw pointers: a forward-mode tangent on a gradient that reaches them would be lost, and the result
// would come back with a derivative of zero.
void refuse_tangents(const variable_list& grads) {
    for (const Tensor& g : grads)
        TORCH_CHECK_NOT_IMPLEMENTED(!g.defined() || !g._fw_grad(/*level=*/0).defined(),
                                    "forward-mode differentiation of the encoding's gradients is not implemented: an incoming gradient has a tangent");
}

// Whether a gradient sent along this edge ends in the .grad of a row-major leaf, which keeps the leaf's layout: autograd
// would bring a level-major gradient into it with a strided copy, at a third of the speed of the library's transpose.  (Any other
// consumer, such as the products of a network's double backward, takes the strided view as it is.)
bool goes_into_row_major_leaf(const torch::autograd::Edge& edge) {
    const auto* const leaf = dynamic_cast<const torch::autograd::AccumulateGrad*>(edge.function.get());
    return leaf != nullptr && leaf->variable.dim() == 2 && leaf->variable.is_contiguous();
}

// Gradients of the slicing w.r.t. the table (0) and the positions (1).  A gradient that nothing in the running pass
// consumes is not computed: the first half of an eikonal loss, autograd.grad(sdf, positions, create_graph=True), runs no
// table scatter.
struct EncodeNode : public Node {
    std::shared_ptr<const Call> call;
    std::shared_ptr<const Slopes> slopes;  // may be null
    void* forward_stream = nullptr;
    // The result counts as saved, as it does in funcs.py: changing it in place, or a second pass through a freed graph, is refused.
    ExpectedVersion result_version;
    bool released = false;

    // A training step on an SDF asks for two table gradients in one pass, through the encoded values and through the
    // position gradient.  The node that meets the second one (EncodeBackNode) runs first, because it names this node as one
    // of its outputs, and leaves it here; this node then computes both in one scatter, where two would each clear, bin
    // and reduce a gradient of the table's size and autograd would add the two.
    std::vector<SecondOrderTerm> second_order;

    std::string name() const override { return "PermutoEncodingBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        released = true;
        slopes.reset();
    }
    std::shared_ptr<const Slopes> kept_slopes() {
        std::lock_guard<std::mutex> lock(mutex_);
        return slopes;
    }
    void check_saved() {
        std::lock_guard<std::mutex> lock(mutex_);
        TORCH_CHECK(!released, torch::autograd::ERR_BACKWARD_TWICE);
        result_version.check("the encoding");
    }

    void leave(SecondOrderTerm term) {
        std::lock_guard<std::mutex> lock(mutex_);
        second_order.push_back(std::move(term));
    }
    std::vector<SecondOrderTerm> take(int task) {
        std::vector<SecondOrderTerm> mine, others;
        std::lock_guard<std::mutex> lock(mutex_);
        for (SecondOrderTerm& t : second_order) (t.task == task ? mine : others).push_back(std::move(t));
        second_order = std::move(others);
        return mine;
    }
    variable_list apply(variable_list&& grads) override;
};

// What the result's grad_fn is: hands its gradient to the EncodeNode.  Hooks on the result live here, so that a pass that
// reaches the EncodeNode from an EncodeBackNode alone does not run them on a gradient that does not exist.
struct ResultNode : public Node {
    std::string name() const override { return "PermutoEncodingResultBackward"; }
    variable_list apply(variable_list&& grads) override { return std::move(grads); }
};

// Gradient of the gradients of the slicing.  Inputs (in the graph's sense): what EncodeNode produced, i.e. the
// gradients w.r.t. the table and w.r.t. the positions; only the path through the latter is differentiated (as in the
// reference, funcs.py:57-72).  Outputs: gradients w.r.t. the upstream gradient, w.r.t. the table, and nothing for the
// slicing, whose node is named so that a pass through both runs it after this one.
struct EncodeBackNode : public Node {
    std::shared_ptr<const Call> call;
    std::shared_ptr<EncodeNode> slicing;
    std::shared_ptr<const Slopes> slopes;     // may be null
    torch::autograd::SavedVariable upstream;  // saved as autograd saves: version checks, hooks, freed with the graph
    ExpectedVersion rows_version;             // of the rows `upstream` is a level-major copy of: changing them is refused all the same

    std::string name() const override { return "PermutoEncodingBackward2"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        upstream.reset_data();
        slopes.reset();
    }
    variable_list apply(variable_list&& grads) override {
        variable_list out(3);
        if (grads.size() < 2 || !grads[1].defined()) return out;
        refuse_tangents(grads);
        Tensor saved;
        Tensor kept;  // held until what reads it has been launched
        {
            std::lock_guard<std::mutex> lock(mutex_);
            saved = upstream.unpack();
            rows_version.check("the upstream gradient");
            if (slopes != nullptr) kept = slopes->usable(*call);
        }
        const Call& c = *call;
        const bool grad_mode = c10::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const c10::DeviceGuard device(c.device());
        const Upstream up = upstream_of(c, saved);  // (a hook may have brought it back in another layout)
        bool want_table = c.want_table && task_should_compute_output(1);
        // (with create_graph the pass stays as it is written: EncodeNode's gradients are then differentiated once more, this one's not)
        if (want_table && !grad_mode && up.row_stride == 0 && task_should_compute_output(2) &&
            current_stream(c.device()) == slicing->forward_stream) {
            slicing->leave({torch::autograd::get_current_graph_task_id(), checked_double_positions_grad(c, grads[1]), up});
            want_table = false;
        }
        bool want_upstream = task_should_compute_output(0);
        if (want_upstream) {
            const bool as_rows = goes_into_row_major_leaf(next_edge(0)) && c.columns() <= 255;
            if (kept.defined()) out[0] = compute_grad_grad(c, kept, checked_double_positions_grad(c, grads[1]), as_rows);
            else if (as_rows) out[0] = compute_grad_grad_rows(c, checked_double_positions_grad(c, grads[1]));
            want_upstream = !out[0].defined();
        }
        if (!want_table && !want_upstream) return out;
        SecondOrder s = compute_double_backward(c, grads[1].detach(), up, want_table, want_upstream);
        if (want_upstream) out[0] = std::move(s.upstream);
        out[1] = std::move(s.table);
        return out;
    }
};

variable_list EncodeNode::apply(variable_list&& grads) {
    variable_list out(2);
    const Call& c = *call;
    refuse_tangents(grads);
    std::vector<SecondOrderTerm> terms = take(torch::autograd::get_current_graph_task_id());
    const bool first_order = !grads.empty() && grads[0].defined();  // undefined: reached through a double backward alone
    const bool want_table = c.want_table && task_should_compute_output(0);
    const bool want_positions = first_order && c.want_positions && task_should_compute_output(1);
    if (!want_table && !want_positions) return out;
    if (!first_order && terms.empty()) return out;
    const bool differentiable = c10::GradMode::is_enabled();
    Upstream up;
    Gradients g;
    ExpectedVersion rows_version;
    std::shared_ptr<const Slopes> slopes_kept;
    {
        at::NoGradGuard no_grad;
        const c10::DeviceGuard device(c.device());
        Tensor kept;  // held until what reads it has been launched
        if (want_positions && (slopes_kept = kept_slopes()) != nullptr && !(kept = slopes_kept->usable(c)).defined()) slopes_kept.reset();
        const SecondOrderTerm* fused = nullptr;
        if (first_order) {
            check_saved();
            up = upstream_of(c, grads[0].detach());
            bool gather_positions = want_positions;
            if (want_positions &&
                (kept.defined() || (differentiable && !want_table && up.row_stride != 0 && c.columns() <= 255))) {
                const bool keep_copy = differentiable || want_table;
                if (differentiable && up.row_stride != 0 && up.values.is_alias_of(grads[0])) rows_version.expect(grads[0]);
                g.positions = compute_positions_backward(c, up, kept, keep_copy);
                gather_positions = false;
            }
            if (want_table || gather_positions) {
                if (want_table && !terms.empty()) fused = &terms.back();
                Gradients more = compute_backward(c, up, want_table, gather_positions, fused);
                g.table = std::move(more.table);
                if (gather_positions) g.positions = std::move(more.positions);
            }
        }
        for (const SecondOrderTerm& t : terms) {
            if (&t == fused || !want_table) continue;
            Tensor more = compute_double_backward(c, t.double_positions_grad, t.upstream, true, false).table;
            if (!more.defined()) continue;  // added into the sparse gradient
            if (g.table.defined()) g.table.add_(more);
            else g.table = std::move(more);
        }
    }
    if (differentiable && first_order) {
        auto back = std::shared_ptr<EncodeBackNode>(new EncodeBackNode(), torch::autograd::deleteNode);
        back->slicing = std::static_pointer_cast<EncodeNode>(shared_from_this());
        back->set_next_edges(torch::autograd::collect_next_edges(grads[0], c.lattice_values));
        back->add_next_edge(torch::autograd::Edge(back->slicing, 0));
        back->call = call;
        back->slopes = std::move(slopes_kept);
        back->upstream = torch::autograd::SavedVariable(up.values, false);
        back->rows_version = std::move(rows_version);
        torch::autograd::set_history(g.table, back);
        torch::autograd::set_history(g.positions, back);
    }
    out[0] = std::move(g.table);
    out[1] = std::move(g.positions);
    return out;
}

// ------------------------------------------------------------------------------------------
// Python

const Tensor& tensor_arg(PyObject* o, const char* name) {
    PENC_REQUIRE(THPVariable_Check(o), name, " must be a torch.Tensor");
    return THPVariable_Unpack(o);
}

// Runs `body` with C++ exceptions turned into Python ones.
template <typename F>
PyObject* guarded(F&& body) {
    try {
        return body();
    } catch (python_error& e) {
        e.restore();
    } catch (const c10::ValueError& e) {
        PyErr_SetString(PyExc_ValueError, e.what_without_backtrace());
    } catch (const c10::OutOfMemoryError& e) {
        PyObject* const torch_module = PyImport_ImportModule("torch");
        PyObject* const type = torch_module != nullptr ? PyObject_GetAttrString(torch_module, "OutOfMemoryError") : nullptr;
        PyErr_SetString(type != nullptr ? type : PyExc_RuntimeError, e.what_without_backtrace());
        Py_XDECREF(type);
        Py_XDECREF(torch_module);
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// The checks of a call, in the order and with the words of _native.EncodingWrapper (reference: src/Encoding.cu:38-45, 57-66).
void prepare_call(Call& c, const Tensor& positions, const Tensor& window) {
    require_f32_gpu(positions, "positions", 2);
    PENC_REQUIRE(positions.size(0) != 0, "Why do we have 0 points");
    PENC_REQUIRE(positions.size(1) == c.pos_dim,
                 "Pos dim for the lattice doesn't correspond with the position of the points. Lattice was initialized with ", c.pos_dim,
                 " and points have pos dim ", positions.size(1));
    const auto type = c.table.scalar_type();
    if (type == at::kHalf || type == at::kBFloat16) {
        PENC_REQUIRE(c.table.is_cuda(), "lattice_values should be in GPU memory. Please call .cuda() on the tensor");
        PENC_REQUIRE(c.table.dim() == 3, "lattice_values should have 3 dimensions, however it has sizes ", c.table.sizes());
        c.table_format = (type == at::kHalf ? PENC_TABLE_FP16 : PENC_TABLE_BF16) | (c.in_cells ? PENC_TABLE_CELLS : 0);
    } else {
        require_f32_gpu(c.table, "lattice_values", 3);
        c.table_format = 0;
    }
    PENC_REQUIRE(c.table.is_contiguous(), "lattice_values must be contiguous (a slot is loaded at a time)");
    PENC_REQUIRE(c.table.size(2) == c.feat, "lattice_values should be nr_levels x capacity x ", c.feat);
    const int64_t levels = c.table.size(0), lim = (int64_t{1} << 31) - 1;
    PENC_REQUIRE(levels <= lim && c.table.size(1) <= lim, "lattice_values is too large");
    require_f32_gpu(c.shift, "random_shift_per_level", 2);
    PENC_REQUIRE(c.shift.size(0) == levels, "Random shift should have the first dimension the same as the nr of resolutions");
    PENC_REQUIRE(c.shift.size(1) == c.pos_dim, "Random shift should have the second dimension the same as the pos dim");
    require_f32_gpu(window, "anneal_window", 1);
    PENC_REQUIRE(window.size(0) == levels, "anneal_window should have the first dimension the same as the nr of resolutions");
    PENC_REQUIRE(c.scale_factor.dim() == 2 && c.scale_factor.size(0) == levels && c.scale_factor.size(1) == c.pos_dim,
                 "scale list should have one entry per level");
    const at::Device dev = positions.device();
    PENC_REQUIRE(c.table.device() == dev, "lattice_values must be on the same device as positions");
    PENC_REQUIRE(c.shift.device() == dev, "random_shift_per_level must be on the same device as positions");
    PENC_REQUIRE(window.device() == dev, "anneal_window must be on the same device as positions");
    if (c.scale_factor.device() != dev) c.scale_factor = c.scale_factor.to(dev);
    c.positions = positions.contiguous();
    c.shift = c.shift.contiguous();
    c.window = window.contiguous();
    c.levels = static_cast<int>(levels);
    c.capacity = static_cast<int>(c.table.size(1));
    c.n = positions.size(0);
    c.extra = api.extra_levels(c.pos_dim, c.feat, c.concat);
}

// A schedule hands its window over in host memory, once per step: copied by a launch, without waiting for the device.
Tensor window_on_device(const Tensor& window, const at::Device& device) {
    constexpr int64_t kMost = 1024;
    if (!window.device().is_cpu() || window.dim() != 1 || window.numel() == 0 || window.numel() > kMost) return window.to(device, at::kFloat);
    const c10::DeviceGuard guard(device);
    // (a graph would replay the window of the step that captured it)
    TORCH_CHECK(c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None,
                "anneal_window is in host memory: a call that is captured in a graph needs it in GPU memory");
    const Tensor host = window.to(at::kFloat).contiguous();
    Tensor out = at::empty({host.numel()}, host.options().device(device));
    check(api.upload(data(host), mutable_data(out), static_cast<int>(host.numel()), current_stream(device)), "upload");
    return out;
}

// Whether something has to see the autograd functions of funcs.py: a functorch transform or a forward-mode tangent, which they
// refuse, a trace, which records them, or a window that requires a gradient, which makes their result require one.
bool needs_autograd_functions(const Tensor& lattice_values, const Tensor& positions, const Tensor& window) {
    return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || torch::jit::tracer::isTracing() ||
           lattice_values._fw_grad(0).defined() || positions._fw_grad(0).defined() || window._fw_grad(0).defined() ||
           (window.requires_grad() && c10::GradMode::is_enabled());
}

// needs_autograd_functions(lattice_values, positions, window) -> whether encode() would return None
PyObject* py_needs_autograd_functions(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    return guarded([&]() -> PyObject* {
        TORCH_CHECK(n_args == 3, "needs_autograd_functions takes 3 arguments");
        return PyBool_FromLong(needs_autograd_functions(tensor_arg(args[0], "lattice_values"), tensor_arg(args[1], "positions"),
                                                        tensor_arg(args[2], "anneal_window")));
    });
}

// encode(lattice_values, table, positions, window, random_shift, scale_factor, pos_dim, nr_feat, concat_points, points_scaling,
//        sparse_owner or None, rows_output, levels_per_pass, max_workspace_bytes or None, fixed_params)
//   -> (N, F(L+E)), or None where the autograd functions are needed
// encode_from_cells: the same from a table that is a copy in cells (table_in_cells)
template <bool kInCells>
PyObject* py_encode(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    return guarded([&]() -> PyObject* {
        TORCH_CHECK(n_args == 15, "encode takes 15 arguments");
        TORCH_CHECK(api.forward != nullptr, "bind() has not been called");
        const Tensor& lattice_values = tensor_arg(args[0], "lattice_values");
        const Tensor& positions = tensor_arg(args[2], "positions");
        Tensor window = tensor_arg(args[3], "anneal_window");
        if (needs_autograd_functions(lattice_values, positions, window)) Py_RETURN_NONE;
        auto call = std::make_shared<Call>();
        Call& c = *call;
        c.lattice_values = lattice_values;
        c.table = tensor_arg(args[1], "lattice_values");
        c.shift = tensor_arg(args[4], "random_shift_per_level");
        c.scale_factor = tensor_arg(args[5], "scale list");
        const at::Device scale_device = c.scale_factor.device();
        c.pos_dim = static_cast<int>(PyLong_AsLong(args[6]));
        c.feat = static_cast<int>(PyLong_AsLong(args[7]));
        c.concat = PyObject_IsTrue(args[8]);
        c.scaling = static_cast<float>(PyFloat_AsDouble(args[9]));
        c.rows_output = PyObject_IsTrue(args[11]);
        c.in_cells = kInCells;
        c.levels_per_pass = PyLong_AsLongLong(args[12]);
        c.max_workspace = args[13] == Py_None ? -1 : PyLong_AsLongLong(args[13]);
        if (PyErr_Occurred()) return nullptr;
        const bool grad_mode = c10::GradMode::is_enabled();
        c.want_table = grad_mode && lattice_values.requires_grad();
        c.want_positions = grad_mode && positions.requires_grad();
        if (c.want_positions) c.hooked = Slopes::hooks_are_set();
        if (args[10] != Py_None && (c.want_table || c.want_positions)) c.sparse_owner = std::make_shared<PyRef>(args[10]);
        Tensor out;
        std::shared_ptr<Slopes> slopes;
        bool captured = false;
        {
            NoGil no_gil;
            at::NoGradGuard no_grad;
            if (positions.is_cuda()) window = window_on_device(window, positions.device());
            prepare_call(c, positions, window);
            const c10::DeviceGuard device(c.device());
            slopes = Slopes::make(c);
            out = compute_forward(c, slopes);
            if (!kInCells && c.table_format != 0) captured = capture_of(static_cast<hipStream_t>(current_stream(c.device()))) != 0;
        }
        if (captured) {  // (a graph reads this copy from now on)
            THPObjectPtr copy(PyLong_FromVoidPtr(const_cast<void*>(c.table.const_data_ptr())));
            if (!copy || PyObject_SetAttrString(args[14], "m_captured_copy", copy.get()) != 0) return nullptr;
        }
        if (c.scale_factor.device() != scale_device) {  // the module was moved: kept where the points are, so that the next call need not copy
            THPObjectPtr moved(THPVariable_Wrap(c.scale_factor));
            if (!moved || PyObject_SetAttrString(args[14], "m_scale_factor", moved.get()) != 0) return nullptr;
        }
        if (c.want_table || c.want_positions) {
            auto node = std::shared_ptr<EncodeNode>(new EncodeNode(), torch::autograd::deleteNode);
            node->set_next_edges(torch::autograd::collect_next_edges(lattice_values, positions));
            node->forward_stream = current_stream(call->device());
            node->call = std::move(call);
            node->slopes = std::move(slopes);
            node->result_version.expect(out);
            auto result = std::shared_ptr<ResultNode>(new ResultNode(), torch::autograd::deleteNode);
            result->add_next_edge(torch::autograd::Edge(node, node->add_input_metadata(out)));
            torch::autograd::set_history(out, result);
        }
        return THPVariable_Wrap(std::move(out));
    });
}

// capture_id(device) -> that of the device's current stream
PyObject* py_capture_id(PyObject*, PyObject* device) {
    return guarded([&]() -> PyObject* {
        const long index = PyLong_AsLong(device);
        if (PyErr_Occurred()) return nullptr;
        return PyLong_FromUnsignedLongLong(capture_of(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(static_cast<c10::DeviceIndex>(index)).stream()));
    });
}

// record_event(device) -> a capsule: what the device's default stream has been given so far; None where the current stream is captured and
// the default stream would wait for it (torch's streams are none of these).  For the device's own streams alone: a fence for the host, which
// an event of torch's has, would stand between the launches before it and after it.
constexpr const char* kEventCapsule = "penc.event";
PyObject* event_of_stream(hipStream_t stream) {
    hipEvent_t event = nullptr;
    C10_HIP_CHECK(hipEventCreateWithFlags(&event, hipEventDisableTiming | hipEventDisableSystemFence));
    const hipError_t recorded = hipEventRecord(event, stream);
    if (recorded != hipSuccess) (void)hipEventDestroy(event);
    C10_HIP_CHECK(recorded);
    return PyCapsule_New(event, kEventCapsule, [](PyObject* capsule) {
        (void)hipEventDestroy(static_cast<hipEvent_t>(PyCapsule_GetPointer(capsule, kEventCapsule)));
    });
}
PyObject* py_record_event(PyObject*, PyObject* device) {
    return guarded([&]() -> PyObject* {
        const auto index = static_cast<c10::DeviceIndex>(PyLong_AsLong(device));
        if (PyErr_Occurred()) return nullptr;
        const c10::DeviceGuard guard(at::Device(at::kCUDA, index));
        const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(index).stream();
        unsigned flags = hipStreamNonBlocking;
        if (capture_of(stream) != 0 && (hipStreamGetFlags(stream, &flags) != hipSuccess || (flags & hipStreamNonBlocking) == 0)) {
            (void)hipGetLastError();
            Py_RETURN_NONE;
        }
        c10::hip::HIPStreamCaptureModeGuard in_a_capture_too{hipStreamCaptureModeRelaxed};
        return event_of_stream(nullptr);
    });
}

// A list of an event of the device's current stream.  Of None where that is the default stream, which is never destroyed nor captured: the event is recorded
// by the first call on another stream, if there is one (a program that trains a 16-bit table makes a copy in every step, and its event 2 to 4 us).
PyObject* event_behind(const at::Device& device) {
    const auto stream = static_cast<hipStream_t>(current_stream(device));
    if (stream == nullptr) return Py_BuildValue("[O]", Py_None);
    const c10::DeviceGuard guard(device);
    THPObjectPtr event(event_of_stream(stream));
    return event ? Py_BuildValue("[N]", event.release()) : nullptr;
}
PyObject* py_event_behind(PyObject*, PyObject* device) {
    return guarded([&]() -> PyObject* {
        const auto index = static_cast<c10::DeviceIndex>(PyLong_AsLong(device));
        return PyErr_Occurred() ? nullptr : event_behind(at::Device(at::kCUDA, index));
    });
}

// rounded_copy(key, table, table_format, points, so_far) -> (key, the table in 16 bits, device, stream, [event], points, [so_far]): what the wrapper keeps of a
// copy it has just made.  (In the interpreter, call by call, 1 us more.)
PyObject* py_rounded_copy(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    return guarded([&]() -> PyObject* {
        TORCH_CHECK(n_args == 5, "rounded_copy takes 5 arguments");
        const Tensor& table = tensor_arg(args[1], "lattice_values");
        const long format = PyLong_AsLong(args[2]);
        if (PyErr_Occurred()) return nullptr;
        Tensor copy;
        {
            NoGil no_gil;
            at::NoGradGuard no_grad;
            copy = table.to(format == PENC_TABLE_FP16 ? at::kHalf : at::kBFloat16);
        }
        THPObjectPtr event(event_behind(copy.device()));
        if (!event) return nullptr;
        return Py_BuildValue("(ONiNNO[O])", args[0], THPVariable_Wrap(copy), static_cast<int>(copy.get_device()),
                             PyLong_FromVoidPtr(current_stream(copy.device())), event.release(), args[3], args[4]);
    });
}

// wait_for_event(event, device): the device's current stream does, or, where it takes part in a capture, which cannot wait for what is outside it, the host
PyObject* py_wait_for_event(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    return guarded([&]() -> PyObject* {
        TORCH_CHECK(n_args == 2, "wait_for_event takes 2 arguments");
        const auto event = static_cast<hipEvent_t>(PyCapsule_GetPointer(args[0], kEventCapsule));
        const auto index = static_cast<c10::DeviceIndex>(PyLong_AsLong(args[1]));
        if (PyErr_Occurred()) return nullptr;
        const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(index).stream();
        if (capture_of(stream) == 0) {
            C10_HIP_CHECK(hipStreamWaitEvent(stream, event, 0));
        } else {
            NoGil no_gil;
            c10::hip::HIPStreamCaptureModeGuard in_a_capture_too{hipStreamCaptureModeRelaxed};
            C10_HIP_CHECK(hipEventSynchronize(event));
        }
        Py_RETURN_NONE;
    });
}

// table_in_cells(table, table_format, pos_dim, max_workspace_bytes or None) -> the table (fp32, or already of that format) as a 16-bit copy in cells;
// None where there is no memory for it, or none for a level of it under the cap
PyObject* py_table_in_cells(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    return guarded([&]() -> PyObject* {
        TORCH_CHECK(n_args == 4, "table_in_cells takes 4 arguments");
        TORCH_CHECK(api.table_cells != nullptr, "bind() has not been called");
        const Tensor& table = tensor_arg(args[0], "lattice_values");
        const int format = static_cast<int>(PyLong_AsLong(args[1])), pos_dim = static_cast<int>(PyLong_AsLong(args[2]));
        const int64_t cap = args[3] == Py_None ? -1 : PyLong_AsLongLong(args[3]);
        if (PyErr_Occurred()) return nullptr;
        const bool fp32 = table.scalar_type() == at::kFloat;
        const auto type = format == PENC_TABLE_FP16 ? at::kHalf : at::kBFloat16;
        PENC_REQUIRE(table.is_cuda() && table.is_contiguous() && table.dim() == 3 && (fp32 || table.scalar_type() == type), "bad table");
        const int levels = static_cast<int>(table.size(0)), capacity = static_cast<int>(table.size(1)), feat = static_cast<int>(table.size(2));
        // (a few levels at a time go through the workspace, which holds at least one)
        int64_t n = static_cast<int64_t>(api.table_cells_workspace_bytes(feat, levels, capacity, format));
        const int64_t one_level = static_cast<int64_t>(api.table_cells_workspace_bytes(feat, 1, capacity, format));
        if (cap >= 0 && n > cap) n = cap;
        if (n < one_level) Py_RETURN_NONE;
        // The library reads a slot at a time.  A table that begins elsewhere, such as a view into flattened parameters, is rounded first.
        const bool in_slots = (reinterpret_cast<uintptr_t>(table.const_data_ptr()) & (std::min<size_t>(feat * table.element_size(), 16) - 1)) == 0;
        const int64_t copy_bytes = 2 * table.numel();
        Tensor cells;
        {
            NoGil no_gil;
            at::NoGradGuard no_grad;
            const c10::DeviceGuard device(table.device());
            Tensor from = table, ws;
            const bool taken = take_optional(table.device(), (in_slots ? 1 : 2) * copy_bytes + n, [&] {
                cells = at::empty(table.sizes(), table.options().dtype(type));
                ws = at::empty({n}, table.options().dtype(at::kByte));
                if (!in_slots) from = table.to(type, /*non_blocking=*/false, /*copy=*/true);
            });
            if (taken)
                check(api.table_cells(pos_dim, feat, levels, capacity, from.const_data_ptr(), fp32 && in_slots ? 0 : format, format,
                                      cells.mutable_data_ptr(), ws.mutable_data_ptr(), static_cast<size_t>(n), current_stream(table.device())),
                      "table_cells");
            else
                cells = Tensor();
        }
        if (!cells.defined()) Py_RETURN_NONE;
        return THPVariable_Wrap(std::move(cells));
    });
}

// adamw_step(param, grad, exp_avg, exp_avg_sq, lr, beta1, beta2, eps, weight_decay, step, skip_zero_gradients)
// adamw_step_sparse(param, grad, exp_avg, exp_avg_sq, touched, lr, beta1, beta2, eps, weight_decay, step): update, clear, unmark
// The kernels write through raw pointers: the in-place change is recorded for autograd's version checks and for the
// 16-bit copy a module keeps of its table.
PyObject* adamw(PyObject* const* args, Py_ssize_t n_args, bool sparse) {
    return guarded([&]() -> PyObject* {
        TORCH_CHECK(n_args == 11, "adamw_step takes 11 arguments");
        TORCH_CHECK(api.adamw_step != nullptr, "bind() has not been called");
        const Tensor& p = tensor_arg(args[0], "param");
        const Tensor& g = tensor_arg(args[1], "grad");
        const Tensor& m = tensor_arg(args[2], "exp_avg");
        const Tensor& v = tensor_arg(args[3], "exp_avg_sq");
        const int first = sparse ? 5 : 4;
        double x[5];
        for (int i = 0; i < 5; ++i) x[i] = PyFloat_AsDouble(args[first + i]);
        const int64_t step = PyLong_AsLongLong(args[first + 5]);
        if (PyErr_Occurred()) return nullptr;
        for (const Tensor* t : {&p, &g, &m, &v})
            TORCH_CHECK(t->is_cuda() && t->scalar_type() == at::kFloat && t->is_contiguous() && t->numel() == p.numel() && t->device() == p.device(),
                        "AdamW: parameter, gradient and moments must be contiguous float32 tensors of one size in the memory of one GPU");
        const c10::DeviceGuard device(p.device());
        void* const stream = current_stream(p.device());
        if (sparse) {
            const Tensor& touched = tensor_arg(args[4], "touched");
            TORCH_CHECK(p.dim() == 3 && touched.is_cuda() && touched.scalar_type() == at::kInt, "AdamW: bad table or map");
            check(api.adamw_step_sparse(mutable_data(p), mutable_data(g), mutable_data(m), mutable_data(v), static_cast<int>(p.size(2)),
                                        static_cast<int>(p.size(0)), static_cast<int>(p.size(1)),
                                        static_cast<uint32_t*>(touched.mutable_data_ptr()), x[0], x[1], x[2], x[3], x[4], step, 1, stream),
                  "adamw_step_sparse");
        } else {
            check(api.adamw_step(mutable_data(p), data(g), mutable_data(m), mutable_data(v), p.numel(), x[0], x[1], x[2], x[3], x[4], step,
                                 PyObject_IsTrue(args[10]), stream),
                  "adamw_step");
        }
        p.unsafeGetTensorImpl()->bump_version();
        Py_RETURN_NONE;
    });
}
PyObject* py_adamw_step(PyObject*, PyObject* const* args, Py_ssize_t n) { return adamw(args, n, false); }
PyObject* py_adamw_step_sparse(PyObject*, PyObject* const* args, Py_ssize_t n) { return adamw(args, n, true); }

// Whether something has to see tensor operations instead of values written through a pointer: a trace records them, a
// torch-dispatch mode (fake tensors, which have no memory, among them), a functorch transform and a torch-function mode (such
// as the one that sets a default device) run something else in their place.
bool operations_are_observed() {
    return torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           at::impl::PythonTorchFunctionTLS::stack_len() > 0;
}

// cosine_window(n, alpha) -> the window of utils.cosine_easing_window, which is what a coarse-to-fine schedule computes in every
// step: 0.5 * (1 + cos(pi * clip(alpha - k, 0, 1) + pi)) in single precision, each operation rounded as torch rounds it (its
// cosine is torch's own); as six tensor operations from the interpreter it cost 18 us, more than the encoding of a small batch.
// None where those operations are observed.
PyObject* py_cosine_window(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    return guarded([&]() -> PyObject* {
        TORCH_CHECK(n_args == 2, "cosine_window takes 2 arguments");
        if (operations_are_observed()) Py_RETURN_NONE;
        const int64_t n = PyLong_AsLongLong(args[0]);
        const float alpha = PyLong_Check(args[1]) ? static_cast<float>(PyLong_AsLongLong(args[1])) : static_cast<float>(PyFloat_AsDouble(args[1]));
        if (PyErr_Occurred()) return nullptr;
        const float pi = static_cast<float>(3.14159265358979323846);
        at::NoGradGuard no_grad;
        Tensor window = at::empty({n}, at::TensorOptions().dtype(at::kFloat));
        float* const w = static_cast<float*>(window.mutable_data_ptr());
        for (int64_t k = 0; k < n; ++k) {
            const float x = std::min(std::max(alpha - static_cast<float>(k), 0.0f), 1.0f);
            const float scaled = pi * x;
            w[k] = scaled + pi;
        }
        window.cos_();
        for (int64_t k = 0; k < n; ++k) w[k] = 0.5f * (w[k] + 1.0f);
        return THPVariable_Wrap(std::move(window));
    });
}

// bind(path): takes the entry points from the library at `path` (already loaded by the Python side; loading it again is a reference).
PyObject* py_bind(PyObject*, PyObject* path) {
    return guarded([&]() -> PyObject* {
        const char* const name = PyUnicode_AsUTF8(path);
        if (name == nullptr) return nullptr;
        void* const lib = dlopen(name, RTLD_NOW | RTLD_LOCAL);
        TORCH_CHECK(lib != nullptr, "cannot load ", name, ": ", dlerror());
#define PENC_FN(fn)                                                                \
    api.fn = reinterpret_cast<decltype(api.fn)>(dlsym(lib, "penc_" #fn));          \
    TORCH_CHECK(api.fn != nullptr, name, " does not export penc_" #fn)
        PENC_FN(status_string);
        PENC_FN(extra_levels);
        PENC_FN(forward);
        PENC_FN(forward_half);
        PENC_FN(forward_rowmajor);
        PENC_FN(forward_rowmajor_workspace_bytes);
        PENC_FN(scatter_workspace_bytes);
        PENC_FN(scatter_useful_bytes);
        PENC_FN(positions_workspace_bytes);
        PENC_FN(backward);
        PENC_FN(backward_half);
        PENC_FN(backward_rowmajor);
        PENC_FN(backward_sparse);
        PENC_FN(backward_both_orders);
        PENC_FN(double_backward_from_positions);
        PENC_FN(double_backward_from_positions_half);
        PENC_FN(double_backward_from_positions_rowmajor);
        PENC_FN(double_backward_from_positions_sparse);
        PENC_FN(adamw_step);
        PENC_FN(adamw_step_sparse);
        PENC_FN(upload);
        PENC_FN(backward_positions_rowmajor);
        PENC_FN(grad_grad_rowmajor);
        PENC_FN(slopes_bytes);
        PENC_FN(forward_cells);
        PENC_FN(forward_cells_workspace_bytes);
        PENC_FN(table_cells);
        PENC_FN(table_cells_workspace_bytes);
        PENC_FN(forward_slopes);
        PENC_FN(backward_positions_slopes);
        PENC_FN(grad_grad_slopes);
#undef PENC_FN
        Py_RETURN_NONE;
    });
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_O, "takes the C ABI from the library at the given path"},
    {"encode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_encode<false>)), METH_FASTCALL, "the encoding of a batch, differentiable"},
    {"encode_from_cells", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_encode<true>)), METH_FASTCALL, "the same from a copy in cells"},
    {"needs_autograd_functions", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_needs_autograd_functions)), METH_FASTCALL,
     "whether a call is for the autograd functions of funcs.py"},
    {"capture_id", py_capture_id, METH_O, "the capture a device's current stream takes part in"},
    {"rounded_copy", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_rounded_copy)), METH_FASTCALL, "a 16-bit copy of a table, as it is kept"},
    {"event_behind", py_event_behind, METH_O, "an event of a device's current stream, where it has to be recorded now"},
    {"record_event", py_record_event, METH_O, "an event of a device's default stream"},
    {"wait_for_event", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_wait_for_event)), METH_FASTCALL, "waits for such an event"},
    {"table_in_cells", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_table_in_cells)), METH_FASTCALL, "a 16-bit copy of a table in cells"},
    {"cosine_window", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_cosine_window)), METH_FASTCALL, "a coarse-to-fine window"},
    {"adamw_step", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_adamw_step)), METH_FASTCALL, "one AdamW step"},
    {"adamw_step_sparse", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_adamw_step_sparse)), METH_FASTCALL,
     "one AdamW step on the touched slot ranges"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_penc_torch", "native autograd path of the encoding", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__penc_torch() {
    // (a key of its own for every copy of this library in the process: the registry ends the process over a name that it has already)
    const std::string key = "penc_slopes " + std::to_string(reinterpret_cast<uintptr_t>(&module));
    if (!c10::FreeHipMemoryCallbacksRegistry()->Has(key))
        c10::FreeHipMemoryCallbacksRegistry()->Register(key, []() -> std::unique_ptr<c10::FreeMemoryCallback> { return std::make_unique<GiveBackSlopes>(); });
    return PyModule_Create(&module);
}

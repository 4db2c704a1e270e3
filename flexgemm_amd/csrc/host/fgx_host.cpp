// Host side of the operators' hot path: tensors in, library calls out.
//
// A convolution call is a handful of kernel launches around buffers from torch's allocator and tables kept on the
// caller's neighbor cache.  Doing that from Python costs more than the kernels do on small inputs (two 64-channel layers of
// 3 716 voxels, forward and backward: 0.69 ms of host time for 0.23 ms of kernels), so it is done here: one call per
// product or cache build, which allocates, fills in the tables the cache does not have yet -- as attributes of the Python
// object, under the names its Python methods use -- and enqueues the kernels through the C ABI of flexgemm_hip.h.
// Policy (algorithm, schedule, which kernel family) stays with the Python callers.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>

#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "../../../include/flexgemm_hip.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// ---- the library -------------------------------------------------------------------------------------------------
#define FGX_HOST_FUNCTIONS(X)                                                                                                     \
    X(fgx_last_error) X(fgx_grid_index_pays) X(fgx_grid_index_walks) X(fgx_subm_neighbor_map_grid_workspace_bytes) X(fgx_subm_cache_grid_workspace_bytes) \
    X(fgx_subm_cache_build_grid_plan) X(fgx_subm_cache_plan_fits) X(fgx_narrow_plan_bytes) X(fgx_cache_post_workspace_bytes) X(fgx_cache_post) X(fgx_spconv_cache_grid_workspace_bytes) X(fgx_spconv_cache_build_grid)                           \
    X(fgx_spconv_out_dims) X(fgx_spconv_out_coords_grid_workspace_bytes) X(fgx_spconv_out_coords_grid_count)                       \
    X(fgx_spconv_out_coords_grid_emit) X(fgx_tile_plan) X(fgx_gather_item_order) X(fgx_gather_item_order_workspace_bytes)          \
    X(fgx_weight_panel_bytes) X(fgx_pack_weight) X(fgx_conv_scratch_bytes) X(fgx_conv_gather_gemm_act_mask)                        \
    X(fgx_conv_gather_gemm_weight_pays) X(fgx_conv_gather_gemm_weight) X(fgx_conv_gemm_pairs_pays) X(fgx_pair_plan_words) X(fgx_pair_plan) X(fgx_conv_gemm_pairs_scratch_bytes) X(fgx_conv_gemm_pairs) X(fgx_conv_gemm_few_pays) X(fgx_conv_gemm_few_mask)                                                             \
    X(fgx_conv_gather_gemm_stream_act_mask) X(fgx_conv_gather_gemm_stream_groups) X(fgx_relu_mask_apply) X(fgx_copy_columns) X(fgx_relu_columns) \
    X(fgx_colsum_scratch_bytes) X(fgx_colsum) X(fgx_wgrad_block_bounds_count) X(fgx_wgrad_block_bounds)                            \
    X(fgx_conv_gemm_stem_pays) X(fgx_conv_gemm_stem) X(fgx_wgrad_stem_pays) X(fgx_wgrad_stem_scratch_bytes) X(fgx_conv_wgrad_stem_cut) X(fgx_wgrad_item_lists_count) X(fgx_wgrad_item_lists) X(fgx_wgrad_scratch_bytes) X(fgx_conv_wgrad_lists)                       \
    X(fgx_wgrad_schedule) X(fgx_wgrad_sweep_fits) X(fgx_conv_wgrad_split_scratch_bytes) X(fgx_conv_wgrad_split)                                                                  \
    X(fgx_wgrad_sweep_plan_bytes) X(fgx_wgrad_sweep_plan) X(fgx_wgrad_sweep_scratch_bytes) X(fgx_conv_wgrad_sweep)                 \
    X(fgx_serialize_encode) X(fgx_serialize_decode) X(fgx_table_lookup)

struct Lib {
#define X(name) decltype(&::name) name = nullptr;
    FGX_HOST_FUNCTIONS(X)
#undef X
} L;

// the Python modules whose switches the calls below read (looked up on every call: tests and users change them)
PyObject* g_impl = nullptr;         // ops.spconv.submanifold_conv3d
PyObject* g_spconv = nullptr;       // ops.spconv
PyObject* g_native = nullptr;       // _native
PyObject* g_table_lookup = nullptr; // _native.table_lookup as it was at binding

void bind(const std::string& path, py::module_ impl, py::module_ spconv, py::module_ native) {
    void* lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    if (lib == nullptr) throw std::runtime_error(std::string("cannot load ") + path + ": " + dlerror());
#define X(name)                                                                                                   \
    L.name = (decltype(L.name))dlsym(lib, #name);                                                                 \
    if (L.name == nullptr) throw std::runtime_error(path + " does not export " #name ": build the package again");
    FGX_HOST_FUNCTIONS(X)
#undef X
    g_impl = impl.release().ptr();
    g_spconv = spconv.release().ptr();
    g_native = native.release().ptr();
    g_table_lookup = PyDict_GetItemString(PyModule_GetDict(g_native), "table_lookup");
}

void check(int rc) {
    if (rc == 0) return;
    const std::string msg = L.fgx_last_error();
    if (rc == -1) throw py::value_error(msg);
    if (rc == -3) {
        PyErr_SetString(PyExc_NotImplementedError, msg.c_str());
        throw py::error_already_set();
    }
    py::object err = py::reinterpret_borrow<py::object>(g_native).attr("NativeError");
    PyErr_SetString(err.ptr(), msg.c_str());
    throw py::error_already_set();
}

// ---- Python attributes ---------------------------------------------------------------------------------------------
PyObject* module_get(PyObject* module, const char* name) {      // borrowed
    PyObject* v = PyDict_GetItemString(PyModule_GetDict(module), name);
    if (v == nullptr) throw py::attribute_error(name);
    return v;
}
long module_int(PyObject* module, const char* name) { return PyLong_AsLong(module_get(module, name)); }

void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// (asking an event would break a capture some other thread is making in the strict mode)
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Whether the stream is being captured, and by which capture.  (The null stream cannot be.)
bool capturing(int64_t stream, unsigned long long* id = nullptr) {
    if (stream == 0) return false;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long which = 0;
    hip_check(hipStreamGetCaptureInfo((hipStream_t)(uintptr_t)stream, &status, &which), "hipStreamGetCaptureInfo");
    if (id != nullptr) *id = which;
    return status != hipStreamCaptureStatusNone;
}

// Everything enqueued on `after` from here on waits for what `before` holds now.
void order_streams(int64_t before, int64_t after) {
    // A stream under capture gives nothing to wait for; whoever began the capture has waited for the stream (torch.cuda.graph waits for the device).
    if (capturing(before)) return;
    const RelaxedCapture relaxed;
    hipEvent_t event = nullptr;
    hip_check(hipEventCreateWithFlags(&event, hipEventDisableTiming), "hipEventCreate");
    hipError_t e = hipEventRecord(event, (hipStream_t)(uintptr_t)before);
    if (e == hipSuccess) {
        e = hipStreamWaitEvent((hipStream_t)(uintptr_t)after, event, 0);
    } else {                                        // (a stream that its owner has destroyed since)
        (void)hipGetLastError();
        e = hipDeviceSynchronize();
    }
    (void)hipEventDestroy(event);
    hip_check(e, "waiting for another stream's tables");
}

// A neighbor cache: a Python object whose instance dictionary holds its tables.
// They are made on the stream of the call that first wants them.  key_made_on is the stream of the newest one; a call on another stream waits for
// that stream, once after every table (kSeenBy).  The order is handed on: whoever makes the newest table has waited for the older ones.  (Another
// thread's call may add tables wherever this one runs Python code: wait_for_tables() after it.)
// Tables that a call makes while its stream is captured are only recorded: nothing fills them before the graph's first replay, which fills
// them anew each time.  They stand apart from the cache's own, for the calls of that capture alone (key_recorded: the capture and its tables).
struct Cache {
    // (names looked up on every call: interned, 10 ns each instead of 50)
    static PyObject* key_recorded() { static PyObject* const k = PyUnicode_InternFromString("_recorded_tables"); return k; }
    static PyObject* key_made_on() { static PyObject* const k = PyUnicode_InternFromString("_tables_made_on"); return k; }
    static constexpr const char* kSeenBy = "_tables_seen_by";
    py::object obj, dict, recorded;
    int64_t stream;
    Cache(py::object o, int64_t stream_) : obj(std::move(o)), dict(obj.attr("__dict__")), stream(stream_) {
        unsigned long long id = 0;
        PyObject* kept = PyDict_GetItem(dict.ptr(), key_recorded());
        if (!capturing(stream, &id)) {
            if (kept != nullptr && PyDict_DelItem(dict.ptr(), key_recorded()) != 0) throw py::error_already_set();
            wait_for_tables();
        } else if (kept != nullptr && PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(kept, 0)) == id) {
            recorded = py::reinterpret_borrow<py::object>(PyTuple_GET_ITEM(kept, 1));
        } else {
            recorded = py::dict();
            const py::tuple entry = py::make_tuple(id, recorded);
            if (PyDict_SetItem(dict.ptr(), key_recorded(), entry.ptr()) != 0) throw py::error_already_set();
        }
    }
    PyObject* find(const char* key) const {         // borrowed, null if absent
        PyObject* v = recorded ? PyDict_GetItemString(recorded.ptr(), key) : nullptr;
        return v != nullptr ? v : PyDict_GetItemString(dict.ptr(), key);
    }
    PyObject* find(const std::string& key) const { return find(key.c_str()); }
    bool has(const char* key) const { return find(key) != nullptr; }
    bool tensor(const std::string& key, Tensor* out) const {
        PyObject* v = find(key);
        if (v == nullptr || !THPVariable_Check(v)) return false;
        *out = THPVariable_Unpack(v);
        return true;
    }
    Tensor need(const char* key) const {        // through the attribute, which may finish what is still in flight
        Tensor t;
        if (tensor(key, &t)) return t;
        return obj.attr(key).cast<Tensor>();
    }
    void set(const std::string& key, py::handle value) const {
        if (PyDict_SetItemString((recorded ? recorded : dict).ptr(), key.c_str(), value.ptr()) != 0) throw py::error_already_set();
        made_here();
    }
    // Calls a Python function that may make tables of this cache.
    template <typename F> auto tables_by(F&& f) const {
        const Py_ssize_t before = PyDict_Size(dict.ptr());
        auto result = f();
        if (PyDict_Size(dict.ptr()) != before) made_here();
        return result;
    }
    void made_here() const {
        if (recorded) return;
        wait_for_tables();
        if (PyDict_GetItemString(dict.ptr(), kSeenBy) != nullptr && PyDict_DelItemString(dict.ptr(), kSeenBy) != 0) throw py::error_already_set();
        if (PyDict_SetItem(dict.ptr(), key_made_on(), py::int_(stream).ptr()) != 0) throw py::error_already_set();
    }
    void wait_for_tables() const {
        if (recorded) return;
        PyObject* made = PyDict_GetItem(dict.ptr(), key_made_on());
        const int64_t made_on = made != nullptr ? PyLong_AsLongLong(made) : stream;
        if (made_on == stream) return;
        PyObject* seen = PyDict_GetItemString(dict.ptr(), kSeenBy);
        const py::int_ mine(stream);
        if (seen != nullptr && PySet_Contains(seen, mine.ptr()) == 1) return;
        {
            const c10::DeviceGuard guard(need("neighbor_map").device());        // (the event belongs to the streams' device, which need not be the current one)
            order_streams(made_on, stream);
        }
        if (seen == nullptr) {
            const py::set fresh;
            if (PyDict_SetItemString(dict.ptr(), kSeenBy, fresh.ptr()) != 0) throw py::error_already_set();
            seen = fresh.ptr();
        }
        if (PySet_Add(seen, mine.ptr()) != 0) throw py::error_already_set();
    }
    void set(const std::string& key, const Tensor& t) const { set(key, py::cast(t)); }
    void drop(const char* key) const {              // (not from what the cache itself is, during a capture)
        if (!recorded && has(key) && PyDict_DelItemString(dict.ptr(), key) != 0) throw py::error_already_set();
    }
};

// ---- buffers ---------------------------------------------------------------------------------------------------------
Tensor make(at::IntArrayRef sizes, at::ScalarType type, const at::Device& dev) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(dev));
}
Tensor workspace(size_t bytes, const at::Device& dev) { return make({(int64_t)(bytes < 256 ? 256 : bytes)}, at::kByte, dev); }
template <typename T = void>
T* ptr(const Tensor& t) {
    if (!t.defined()) return nullptr;
    if (!t.is_contiguous()) throw py::value_error("a strided view was about to be passed as a plain pointer");    // the kernels assume dense rows
    return (T*)t.data_ptr();
}
fgx_stream_t as_stream(int64_t s) { return (fgx_stream_t)(uintptr_t)s; }
// handle of the current stream of the tensor's device
int64_t stream_of(const Tensor& t) { return (int64_t)(uintptr_t)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// ---- the segment table on its way to the host ------------------------------------------------------------------------
// The pair lists' segment table is written to a pinned block by the kernel that fills the lists; the event behind it tells
// when it has arrived.  Blocks are kept for the next cache (at most kIdleBlocks of them; one that may still be written is
// not handed out), the rest is freed.
struct SegBlock {
    uint32_t* words = nullptr;
    hipEvent_t event = nullptr;
    int device = -1;
};
constexpr size_t kIdleBlocks = 64, kSegWords = 64;
std::mutex g_blocks_mutex;
std::vector<SegBlock> g_idle_blocks;

SegBlock take_block(int device) {
    const RelaxedCapture relaxed;
    {
        std::lock_guard<std::mutex> lock(g_blocks_mutex);
        for (size_t i = 0; i < g_idle_blocks.size(); ++i)
            if (g_idle_blocks[i].device == device && hipEventQuery(g_idle_blocks[i].event) == hipSuccess) {
                const SegBlock b = g_idle_blocks[i];
                g_idle_blocks[i] = g_idle_blocks.back();
                g_idle_blocks.pop_back();
                return b;
            }
    }
    (void)hipGetLastError();        // (a query of an event still ahead leaves its answer behind as an error)
    SegBlock b;
    b.device = device;
    hip_check(hipHostMalloc((void**)&b.words, kSegWords * sizeof(uint32_t), hipHostMallocPortable | hipHostMallocMapped), "hipHostMalloc");
    hip_check(hipEventCreateWithFlags(&b.event, hipEventDisableTiming), "hipEventCreate");
    return b;
}

void give_block(const SegBlock& b) {
    {
        std::lock_guard<std::mutex> lock(g_blocks_mutex);
        if (g_idle_blocks.size() < kIdleBlocks) {
            g_idle_blocks.push_back(b);
            return;
        }
    }
    const RelaxedCapture relaxed;
    (void)hipEventSynchronize(b.event);
    (void)hipEventDestroy(b.event);
    (void)hipHostFree(b.words);
}

class SegHost {
public:
    SegHost(int device, int count) : block_(take_block(device)), count_(count) {}
    ~SegHost() { give_block(block_); }
    SegHost(const SegHost&) = delete;
    SegHost& operator=(const SegHost&) = delete;
    uint32_t* words() { return block_.words; }
    void record(fgx_stream_t s) { hip_check(hipEventRecord(block_.event, (hipStream_t)s), "hipEventRecord"); }
    void synchronize() {
        py::gil_scoped_release nogil;
        hip_check(hipEventSynchronize(block_.event), "hipEventSynchronize");
    }
    py::list tolist() const {
        py::list out;
        for (int i = 0; i < count_; ++i) out.append(py::int_(block_.words[i]));
        return out;
    }

private:
    SegBlock block_;
    int count_;
};

// ---- neighbor caches ---------------------------------------------------------------------------------------------------
// The layer a cache is built for.
struct Layer {
    int code;                       // dtype (-1: one the kernels do not take)
    int64_t ci, co;
    bool record, input_grad, weight_grad, splitk;
};
struct Needs {
    bool order = true, lists = true, plan = false;          // plan: the narrow layers', at the first product
};

bool schedules_are_ours();
std::string narrow_mode() { return py::reinterpret_borrow<py::object>(module_get(g_spconv, "NARROW_RESIDENT")).cast<std::string>(); }

// Few voxels under a small weight, in one launch.  (A map as long as the private row order starts at is not one of few voxels: lowering that limit
// asks for the order.)
bool few_pays(int code, int64_t n, int ci, int co, int v) {
    return L.fgx_conv_gemm_few_pays(code, (size_t)n, ci, co, v) && n < module_int(g_impl, "LOCALITY_MIN_ROWS");
}

// Output columns that the kernels of whole 16-byte pieces (resident rows, first layers) multiply for `cols` 16-bit ones: the columns, or over many
// rows those filled up to a multiple of 8 and cut afterwards, a pass over the output and two or three small copies.  Before and now, us:
// 11 -> 11 channels, cache and one layer, 1.84 million voxels 688 398;  64 -> 19, then three of 19, 1.30 million 1296 688;  27 -> 27, 229 217 voxels, cache
// and one layer 144 94, trained 307 203 where the host keeps up with the copies' launches and 307 310 where it does not (kept 183, 134 and 232);
// 6 -> 41, fresh and kept, 73 461 voxels 62 49 and 43 31, trained 109 117 and 88 96, 229 217 voxels 180 128 and 102 98.
int whole_columns(int cols, int64_t n) { return cols % 8 == 0 || n < (cols > 32 ? 131072 : 393216) ? cols : (cols + 7) / 8 * 8; }

// What of the mask order and the pair lists the kernels of this layer read (a guess that errs towards "all of it": what a pass finds missing
// it makes).  The resident-row kernels walk the cells of the index, first layers the map, the products over pairs a plan of
// their own; so of the tables of 2 667 120 voxels under 32 channels 0.26 ms of sorts and 0.19 ms of lists were never read, of 434 000 voxels under a
// first layer 0.05 and 0.03 of 0.27.
Needs layer_needs(const Layer& l, int64_t n, int v, bool walks) {
    Needs needs;
    if (!schedules_are_ours()) return needs;
    const int es = l.code == FGX_F32 ? 4 : 2, align = 16 / es;
    const int ci = (int)((l.ci + align - 1) / align * align), co = (int)((l.co + align - 1) / align * align);
    const int out_cols = es == 2 ? whole_columns((int)l.co, n) : (int)l.co, in_cols = es == 2 ? whole_columns((int)l.ci, n) : (int)l.ci;
    const bool resident = es == 2 && walks && v <= 27 && ci <= 32 && out_cols <= 32 && out_cols % 8 == 0 && n >= module_int(g_impl, "NARROW_RESIDENT_MIN_ROWS") &&
                          narrow_mode() != "off";
    const bool forward = resident || L.fgx_conv_gemm_stem_pays(l.code, 0, (size_t)n, ci, out_cols, v) ||
                         (l.splitk && (L.fgx_conv_gemm_pairs_pays(l.code, 0, (size_t)n, ci, (int)l.co, v) ||
                                       few_pays(l.code, n, ci, (int)l.co, v)));
    const bool backward = !l.record || !l.input_grad || (resident && in_cols % 8 == 0) || L.fgx_conv_gemm_stem_pays(l.code, 1, (size_t)n, co, in_cols, v) ||
                          (l.splitk && L.fgx_conv_gemm_pairs_pays(l.code, 1, (size_t)n, (int)l.ci, co, v));
    needs.order = !(forward && backward);
    needs.plan = resident && n * 82 + 10752 < 0xFF000000ll && n * ci * 2 < 0xFF000000ll;        // (what _narrow_applies asks)
    needs.lists = l.record && l.weight_grad && !resident && !L.fgx_wgrad_stem_pays(l.code, (size_t)n, ci, co, v);
    return needs;
}

// The pair lists' length is waited for, which a capture does not allow: refused before the cache is touched.
void refuse_lists_in_capture(int64_t stream) {
    if (capturing(stream))
        throw std::runtime_error("the pair lists of a neighbor cache cannot be made while the stream is being captured; run the layer once before the capture");
}

// The mask order and / or the pair lists of a cache that was built without them.
void cache_post(const Cache& c, bool order, bool lists) {
    if (lists) refuse_lists_in_capture(stream_of(c.need("neighbor_map")));
    const Tensor nmap = c.need("neighbor_map"), gray = c.need("gray_code"), binary = c.need("_binary_code");
    const at::Device dev = nmap.device();
    const c10::DeviceGuard guard(dev);
    const int64_t stream = stream_of(nmap), n = nmap.size(0);
    const int v = (int)nmap.size(1);
    Tensor sorted, seg, sig_i, sig_o;
    std::unique_ptr<SegHost> host;
    if (order) sorted = make({n}, at::kLong, dev);
    if (lists) {
        seg = make({v + 1}, at::kUInt32, dev);
        sig_i = make({n * v}, at::kUInt32, dev);
        sig_o = make({n * v}, at::kUInt32, dev);
        host = std::make_unique<SegHost>(dev.index(), v + 1);
    }
    Tensor ws = workspace(L.fgx_cache_post_workspace_bytes((size_t)n, v, lists), dev);
    check(L.fgx_cache_post(ptr<uint32_t>(nmap), ptr<int32_t>(gray), ptr<int32_t>(binary), (size_t)n, v, lists, ptr(ws), (size_t)ws.numel(),
                           ptr<int64_t>(sorted), ptr<uint32_t>(seg), ptr<uint32_t>(sig_i), ptr<uint32_t>(sig_o), host ? host->words() : nullptr,
                           as_stream(stream)));
    if (order) {
        c.set("sorted_idx", sorted);
        c.drop("_order_left_out");
    }
    if (lists) {
        host->record(as_stream(stream));
        const py::object arriving = py::cast(std::move(host));
        c.set("valid_signal_seg", seg);
        c.set("_pending_pairs", py::make_tuple(sig_i, sig_o, arriving, arriving));
        c.drop("_lists_left_out");
    }
}

// Tables of a submanifold convolution through the grid index, or None where it does not apply:
// (neighbor_map, gray, binary, order, walk, seg, sig_i, sig_o, SegHost, plan), the four before the plan None without gradients; walk: the rows in the
// order of the index's cells, for the plan of narrow layers, or None; last that plan, where the layer wants it at once, or None.  layer (dtype code, ci, co, record, input_grad, weight_grad, splitk):
// the layer that asks, whose kernels may read neither the order nor the lists; those are None then.
py::object subm_cache(const Tensor& coords, const std::vector<int>& geom, bool needs_grad, bool forced, size_t max_pair_bytes,
                      const c10::optional<std::tuple<int, int64_t, int64_t, bool, bool, bool, bool>>& layer) {
    const int64_t stream = stream_of(coords);
    const size_t n = (size_t)coords.size(0);
    const int B = geom[0], W = geom[1], H = geom[2], D = geom[3], V = geom[4] * geom[5] * geom[6];
    if (n == 0 || V > 32 || n * (size_t)V >= 0xFFFFFFFFull || (needs_grad && n * (size_t)V * 8 > max_pair_bytes)) return py::none();
    if (needs_grad && capturing(stream)) return py::none();        // (nothing may wait for the segment table inside a capture)
    if (!L.fgx_grid_index_pays(n, B, W, H, D) && !(forced && L.fgx_subm_neighbor_map_grid_workspace_bytes(n, B, W, H, D))) return py::none();
    const at::Device dev = coords.device();
    const c10::DeviceGuard guard(dev);
    const int64_t rows = (int64_t)n, slots = rows * V;
    const bool walks = rows >= module_int(g_impl, "NARROW_RESIDENT_MIN_ROWS") && L.fgx_grid_index_walks(n, B, W, H, D);
    Needs needs;
    if (layer && std::get<0>(*layer) >= 0) {
        const auto& [code, ci, co, record, input_grad, weight_grad, splitk] = *layer;
        needs = layer_needs(Layer{code, ci, co, record, input_grad, weight_grad, splitk}, rows, V, walks);
    }
    const bool lists = needs_grad && needs.lists;
    Tensor nmap = make({rows, V}, at::kUInt32, dev), gray = make({rows}, at::kInt, dev), binary = make({rows}, at::kInt, dev);
    Tensor order, seg, sig_i, sig_o;
    std::unique_ptr<SegHost> host;
    if (needs.order) order = make({rows}, at::kLong, dev);
    if (lists) {
        seg = make({V + 1}, at::kUInt32, dev);
        sig_i = make({slots}, at::kUInt32, dev);
        sig_o = make({slots}, at::kUInt32, dev);
        host = std::make_unique<SegHost>(dev.index(), V + 1);
    }
    Tensor walk;
    if (walks) walk = make({rows}, at::kUInt32, dev);
    // (none is made inside a capture: it would be made again on every replay)
    Tensor plan;
    if (needs.plan && walks && V == 27 && L.fgx_subm_cache_plan_fits(n, B, W, H, D, geom[4], geom[5], geom[6], geom[9]) && !capturing(stream))
        plan = make({(int64_t)L.fgx_narrow_plan_bytes(n, V)}, at::kByte, dev);
    Tensor ws = workspace(L.fgx_subm_cache_grid_workspace_bytes(n, B, W, H, D, V, lists), dev);
    check(L.fgx_subm_cache_build_grid_plan(ptr<int32_t>(coords), n, B, W, H, D, geom[4], geom[5], geom[6], geom[7], geom[8], geom[9], lists,
                                      ptr(ws), (size_t)ws.numel(), ptr<uint32_t>(nmap), ptr<int32_t>(gray), ptr<int32_t>(binary),
                                      ptr<int64_t>(order), ptr<uint32_t>(seg), ptr<uint32_t>(sig_i), ptr<uint32_t>(sig_o),
                                      host ? host->words() : nullptr, ptr<uint32_t>(walk), ptr(plan), as_stream(stream)));
    const py::object plan_out = plan.defined() ? py::cast(plan) : py::none();
    py::object walk_out = walk.defined() ? py::cast(walk) : py::none();
    const py::object order_out = order.defined() ? py::cast(order) : py::none();
    if (!host) return py::make_tuple(nmap, gray, binary, order_out, walk_out, py::none(), py::none(), py::none(), py::none(), plan_out);
    host->record(as_stream(stream));
    return py::make_tuple(nmap, gray, binary, order_out, walk_out, seg, sig_i, sig_o, std::move(host), plan_out);
}

bool conv_grids_pay(size_t n_in, size_t n_out, int B, const int* in, const int* out, bool with_bwd) {
    return L.fgx_grid_index_pays(n_in, B, in[0], in[1], in[2]) && (!with_bwd || L.fgx_grid_index_pays(n_out, B, out[0], out[1], out[2]));
}

// geom: B, W, H, D, kernel, stride, padding, dilation.  The dictionary of a generic convolution's tables, or None.
py::object spconv_cache(const Tensor& coords, const Tensor& out_coords, const std::vector<int>& g, bool needs_grad, bool bwd_order,
                        size_t max_pair_bytes) {
    const int64_t stream = stream_of(coords);
    const size_t m = (size_t)coords.size(0), l = (size_t)out_coords.size(0);
    const int V = g[4] * g[5] * g[6];
    if (m == 0 || l == 0 || V > 32 || l * (size_t)V >= 0xFFFFFFFFull || (needs_grad && l * (size_t)V * 8 > max_pair_bytes)) return py::none();
    if (needs_grad && capturing(stream)) return py::none();        // (as in subm_cache)
    int out[3];
    check(L.fgx_spconv_out_dims(g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8], g[9], g[10], g[11], g[12], g[13], g[14], g[15], &out[0], &out[1], &out[2]));
    if (out[0] < 1 || out[1] < 1 || out[2] < 1 || !conv_grids_pay(m, l, g[0], &g[1], out, needs_grad)) return py::none();
    const at::Device dev = coords.device();
    const c10::DeviceGuard guard(dev);
    const int64_t rows = (int64_t)l;
    Tensor nmap = make({rows, V}, at::kUInt32, dev), gray = make({rows}, at::kInt, dev), binary = make({rows}, at::kInt, dev);
    Tensor order = make({rows}, at::kLong, dev), nmap_bwd, seg, sig_i, sig_o, gray_bwd, order_bwd;
    std::unique_ptr<SegHost> host;
    if (needs_grad) {
        nmap_bwd = make({(int64_t)m, V}, at::kUInt32, dev);
        seg = make({V + 1}, at::kUInt32, dev);
        sig_i = make({rows * V}, at::kUInt32, dev);
        sig_o = make({rows * V}, at::kUInt32, dev);
        host = std::make_unique<SegHost>(dev.index(), V + 1);
        if (bwd_order) {
            gray_bwd = make({(int64_t)m}, at::kInt, dev);
            order_bwd = make({(int64_t)m}, at::kLong, dev);
        }
    }
    Tensor ws = workspace(L.fgx_spconv_cache_grid_workspace_bytes(m, l, g[0], g[1], g[2], g[3], out[0], out[1], out[2], V, needs_grad,
                                                                  order_bwd.defined()), dev);
    check(L.fgx_spconv_cache_build_grid(ptr<int32_t>(coords), m, ptr<int32_t>(out_coords), l, g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8],
                                        g[9], g[10], g[11], g[12], g[13], g[14], g[15], ptr(ws), (size_t)ws.numel(), ptr<uint32_t>(nmap),
                                        ptr<int32_t>(gray), ptr<int32_t>(binary), ptr<int64_t>(order), ptr<uint32_t>(nmap_bwd), ptr<uint32_t>(seg),
                                        ptr<uint32_t>(sig_i), ptr<uint32_t>(sig_o), host ? host->words() : nullptr, ptr<int32_t>(gray_bwd),
                                        ptr<int64_t>(order_bwd), as_stream(stream)));
    py::dict t;
    t["nmap"] = nmap;
    t["gray"] = gray;
    t["order"] = order;
    if (needs_grad) {
        host->record(as_stream(stream));
        t["nmap_bwd"] = nmap_bwd;
        if (bwd_order) {
            t["gray_bwd"] = gray_bwd;
            t["order_bwd"] = order_bwd;
        }
        t["pairs"] = py::dict(py::arg("seg") = seg, py::arg("pending") = py::make_tuple(sig_i, sig_o, py::cast(std::move(host))));
    }
    return std::move(t);
}

// Output coordinates in (b, x, y, z) order through the bit map of the output grid, or None where it does not apply.
py::object out_coords(const Tensor& coords, const std::vector<int>& g) {
    const int64_t stream = stream_of(coords);
    if (capturing(stream)) return py::none();              // (the count is waited for)
    const size_t m = (size_t)coords.size(0);
    int out[3];
    check(L.fgx_spconv_out_dims(g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8], g[9], g[10], g[11], g[12], g[13], g[14], g[15], &out[0], &out[1], &out[2]));
    if (m * (size_t)g[4] * g[5] * g[6] >= (size_t)1 << 30 || !L.fgx_grid_index_pays(m, g[0], out[0], out[1], out[2])) return py::none();
    const at::Device dev = coords.device();
    const c10::DeviceGuard guard(dev);
    Tensor ws = workspace(L.fgx_spconv_out_coords_grid_workspace_bytes(g[0], out[0], out[1], out[2]), dev);
    SegHost host(dev.index(), 2);           // the number of coordinates, as one 64-bit word
    check(L.fgx_spconv_out_coords_grid_count(ptr<int32_t>(coords), m, g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8], g[9], g[10], g[11],
                                             g[12], g[13], g[14], g[15], ptr(ws), (size_t)ws.numel(), (uint64_t*)host.words(), as_stream(stream)));
    host.record(as_stream(stream));
    host.synchronize();                     // the one wait of the host: sizes the result
    uint64_t total;
    memcpy(&total, host.words(), sizeof(total));
    Tensor result = make({(int64_t)total, 4}, at::kInt, dev);
    check(L.fgx_spconv_out_coords_grid_emit(ptr(ws), g[0], out[0], out[1], out[2], (size_t)total, ptr<int32_t>(result), as_stream(stream)));
    return py::cast(result);
}

// ---- tile tables -----------------------------------------------------------------------------------------------------
struct Tiles {
    Tensor order, code, plan_seg, plan_idx, plan_band;
    std::string plan_key;
};

// Row order and tile masks of the masked schedule for tiles of `block` rows (own_order: the kernels' own row order).
void tile_codes(const Cache& c, int block, bool own_order, int64_t stream, Tiles* t, bool for_plan) {
    t->order = c.need(own_order ? "_tile_order" : "sorted_idx");
    const std::string key = (own_order ? "_tile_code_" : "_mask_code_") + std::to_string(block);
    if (c.tensor(key, &t->code) || for_plan) return;        // (the plan's call makes the masks on its way)
    const Tensor gray = c.need("gray_code");
    const int64_t n = gray.size(0);
    t->code = make({(n + block - 1) / block}, at::kInt, gray.device());
    check(L.fgx_tile_plan(ptr<int32_t>(gray), ptr<int64_t>(t->order), nullptr, (size_t)n, 1, block, 0, ptr<int32_t>(t->code), nullptr, nullptr,
                          nullptr, nullptr, 1, 1, 1, nullptr, nullptr, as_stream(stream)));
    c.set(key, t->code);
}

// How the tiles of a streaming GEMM are dealt: by cost ("balanced") or in the kernel's own order.
// The locality order of short-row layers lives on neighboring tiles sharing an XCD (dealing them by cost alone: 0.32 -> 0.42
// ms per launch at C = 32); with rows of 512 bytes and more balance wins whatever the number of tiles (-6 % per launch at
// C = 256, -8 % at C = 1024); with shorter rows it wins while a workgroup has few tiles (C = 128, forward: 143 616 voxels
// 0.120 -> 0.101 ms, 252 392 voxels 0.179 -> 0.155, 577 592 voxels 0.342 -> 0.320; 669 288 voxels, 10 rounds of items, and
// 1 026 536 voxels, 16 rounds: no change).  With at most one item per workgroup there is nothing to even out; from there on
// the dealt order pays (forward at 64 160 voxels: C = 256, two rounds of items, 0.158 -> 0.141 ms; C = 512, four rounds, 0.550
// -> 0.512 ms; 15 192 voxels C = 1024, two rounds, 0.601 -> 0.568 ms).
bool deal_items(const std::string& plan_key, int64_t tiles, int col_tiles, int groups, int slabs) {
    std::string mode = py::reinterpret_borrow<py::object>(module_get(g_spconv, "GEMM_ITEM_ORDER")).cast<std::string>();
    const int64_t items = tiles * col_tiles;
    if (mode == "auto") {
        const bool few_rounds = items <= module_int(g_impl, "ITEM_ORDER_ANY_ROW_MAX_ROUNDS") * groups;
        mode = (slabs >= 4 || few_rounds) && plan_key.rfind("_plan_t_", 0) != 0 ? "balanced" : "default";
    }
    if (mode == "default" || items <= module_int(g_impl, "ITEM_ORDER_MIN_ROUNDS") * groups || groups > 1024 || items >= 0x7FFFFFFF) return false;
    if (mode != "balanced") throw py::value_error("unknown GEMM_ITEM_ORDER '" + mode + "'; expected 'auto', 'balanced' or 'default'");
    return true;
}

std::string items_key(const std::string& plan_key, int col_tiles, int groups, int slabs) {
    return "_items_" + plan_key + "_" + std::to_string(col_tiles) + "_" + std::to_string(groups) + "_" + std::to_string(slabs);
}

Tensor item_order(const Cache& c, const std::string& plan_key, const Tensor& code, int col_tiles, int groups, int slabs, int64_t stream) {
    Tensor item_at;
    if (!deal_items(plan_key, code.size(0), col_tiles, groups, slabs)) return item_at;
    const std::string key = items_key(plan_key, col_tiles, groups, slabs);
    if (c.tensor(key, &item_at)) return item_at;
    const size_t nb = (size_t)code.size(0);
    item_at = make({code.size(0) * col_tiles}, at::kInt, code.device());
    Tensor ws = workspace(L.fgx_gather_item_order_workspace_bytes(nb, col_tiles), code.device());
    check(L.fgx_gather_item_order(ptr<int32_t>(code), nb, col_tiles, slabs, groups, ptr(ws), (size_t)ws.numel(), ptr<uint32_t>(item_at), as_stream(stream)));
    c.set(key, item_at);
    return item_at;
}

// The gather plan for tiles of `block` rows (dense: rows in their natural order, every tile all offsets), and with
// col_tiles > 0 the item order of a launch over it; whatever is missing is made in one call.
Tiles gather_plan(const Cache& c, int block, bool own_order, bool dense, int col_tiles, int groups, int slabs, Tensor* item_at, int64_t stream) {
    Tiles t;
    if (dense) {
        const py::tuple oc = c.tables_by([&] { return py::tuple(c.obj.attr("_dense_tile_tables")(block)); });
        t.order = oc[0].cast<Tensor>();
        t.code = oc[1].cast<Tensor>();
        t.plan_key = "_plan_d_" + std::to_string(block);
    } else {
        tile_codes(c, block, own_order, stream, &t, true);
        t.plan_key = std::string(own_order ? "_plan_t_" : "_plan_m_") + std::to_string(block);
    }
    PyObject* kept = c.find(t.plan_key);
    if (kept != nullptr) {
        py::tuple p = py::reinterpret_borrow<py::tuple>(kept);
        t.plan_seg = p[0].cast<Tensor>();
        t.plan_idx = p[1].cast<Tensor>();
        t.plan_band = p[2].cast<Tensor>();
        if (item_at != nullptr) *item_at = item_order(c, t.plan_key, t.code, col_tiles, groups, slabs, stream);
        return t;
    }
    const Tensor nmap = c.need("neighbor_map");
    const at::Device dev = nmap.device();
    const int64_t n = nmap.size(0), v = nmap.size(1), nb = (n + block - 1) / block;
    const bool have_codes = t.code.defined();
    Tensor gray;
    if (!have_codes) {
        gray = c.need("gray_code");
        t.code = make({nb}, at::kInt, dev);
    }
    t.plan_seg = make({nb + 1}, at::kInt, dev);
    const int64_t rows = nb * std::min<int64_t>(v, 32);       // the bound (every offset in every tile): no wait for the exact count
    t.plan_idx = make({rows, block}, at::kUInt32, dev);
    t.plan_band = make({rows}, at::kUInt32, dev);
    Tensor items_ws;
    if (item_at != nullptr && deal_items(t.plan_key, nb, col_tiles, groups, slabs)) {
        *item_at = make({nb * col_tiles}, at::kInt, dev);
        items_ws = workspace(L.fgx_gather_item_order_workspace_bytes((size_t)nb, col_tiles), dev);
    }
    check(L.fgx_tile_plan(ptr<int32_t>(gray), ptr<int64_t>(t.order), ptr<uint32_t>(nmap), (size_t)n, (int)v, block, have_codes, ptr<int32_t>(t.code),
                          nullptr, ptr<int32_t>(t.plan_seg), ptr<uint32_t>(t.plan_idx), ptr<uint32_t>(t.plan_band), col_tiles > 0 ? col_tiles : 1,
                          slabs > 0 ? slabs : 1, groups > 0 ? groups : 1, ptr<uint32_t>(items_ws),
                          items_ws.defined() ? ptr<uint32_t>(*item_at) : nullptr, as_stream(stream)));
    if (!have_codes) c.set((own_order ? "_tile_code_" : "_mask_code_") + std::to_string(block), t.code);
    c.set(t.plan_key, py::make_tuple(t.plan_seg, t.plan_idx, t.plan_band));
    if (items_ws.defined()) c.set(items_key(t.plan_key, col_tiles, groups, slabs), *item_at);
    return t;
}

// ---- products --------------------------------------------------------------------------------------------------------
struct Sched {
    int tile_rows, tile_cols, slab_bytes, splitk, block_rows, stream;
};

Sched read_schedule(py::handle s) {
    Py_buffer view;
    if (PyObject_GetBuffer(s.ptr(), &view, PyBUF_SIMPLE) != 0) throw py::error_already_set();
    Sched out;
    const bool fits = view.len == (Py_ssize_t)sizeof(out);
    if (fits) memcpy(&out, view.buf, sizeof(out));
    PyBuffer_Release(&view);
    if (!fits) throw py::value_error("not a schedule");
    return out;
}

void mark(const char* name, const char* phase) {
    PyObject* hook = PyDict_GetItemString(PyModule_GetDict(g_native), "EVENT_HOOK");
    if (hook != nullptr && hook != Py_None) py::reinterpret_borrow<py::object>(hook)(name, phase);
}

int dtype_code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kHalf: return FGX_F16;
        case at::kBFloat16: return FGX_BF16;
        case at::kFloat: return FGX_F32;
        default: throw py::type_error("unsupported feature dtype; expected float16, bfloat16 or float32");
    }
}

int ceil_div(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

// The schedule of a pass and shape (fgx_table_lookup; answers are pure functions of the key and remembered).  Python's
// table_lookup is asked instead when somebody has replaced it: that is how schedules are forced.
py::object python_schedule(int pass, const Tensor& like, int64_t n, int ci, int co, int v) {
    return py::reinterpret_borrow<py::object>(module_get(g_native, "table_lookup"))(
        pass, py::cast(like).attr("dtype"), n, ci, co, v);
}

// Nobody has replaced the schedules: a forced one names the kernels that take schedules, not the first layers'.
bool schedules_are_ours() { return module_get(g_native, "table_lookup") == g_table_lookup; }

Sched schedule(int pass, const Tensor& like, int64_t n, int ci, int co, int v) {
    if (!schedules_are_ours()) return read_schedule(python_schedule(pass, like, n, ci, co, v));
    struct Key {
        int pass, code, ci, co, v;
        int64_t n;
        bool operator==(const Key& o) const { return pass == o.pass && code == o.code && ci == o.ci && co == o.co && v == o.v && n == o.n; }
    };
    struct Hash {
        size_t operator()(const Key& k) const {
            uint64_t h = (uint64_t)k.n * 0x9E3779B97F4A7C15ull;
            for (int x : {k.pass, k.code, k.ci, k.co, k.v}) h = (h ^ (uint64_t)x) * 0x9E3779B97F4A7C15ull + (h >> 29);
            return (size_t)h;
        }
    };
    static std::unordered_map<Key, Sched, Hash> known;      // (guarded by the interpreter lock, like all callers here)
    const Key key{pass, dtype_code(like), ci, co, v, n};
    auto it = known.find(key);
    if (it == known.end()) {
        fgx_schedule got;
        static_assert(sizeof(got) == sizeof(Sched), "the schedule's fields");
        check(L.fgx_table_lookup(pass, key.code, (size_t)n, ci, co, v, &got));
        Sched s;
        memcpy(&s, &got, sizeof(s));
        if (known.size() > 4096) known.clear();
        it = known.emplace(key, s).first;
    }
    return it->second;
}

bool aligned(const Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }

py::object impl_function(const char* name) { return py::reinterpret_borrow<py::object>(module_get(g_impl, name)); }

// Whether the resident-row kernels for narrow layers could run at all; the Python policy decides when they do.
bool narrow_shape(const Cache& c, int es, int k, int cols, int v, int64_t n) {
    if (es != 2 || k < 8 || k > 32 || k % 8 || cols < 8 || cols > 32 || cols % 8 || v > 27) return false;
    return c.has("_narrow_plan_buf") || n >= module_int(g_impl, "NARROW_RESIDENT_MIN_ROWS") ||
           py::reinterpret_borrow<py::object>(module_get(g_spconv, "NARROW_RESIDENT")).cast<std::string>() != "auto";
}

// A contiguous tensor of rows of `cols` elements as one of `sizes` with rows of `out_cols`: filled up with zeros, or cut.
Tensor copy_columns(const Tensor& t, int64_t rows, int64_t cols, at::IntArrayRef sizes, int64_t out_cols, int64_t stream) {
    Tensor out = make(sizes, t.scalar_type(), t.device());
    if (rows > 0) check(L.fgx_copy_columns((int)t.element_size(), ptr(t), (size_t)rows, (int)cols, ptr(out), (int)out_cols, as_stream(stream)));
    return out;
}

// `dim` (the last one, or the first of a contiguous tensor) filled up with zeros to a multiple
Tensor pad_to(const Tensor& t, int64_t dim, int64_t multiple, int64_t stream) {
    const int64_t size = t.size(dim), padded = (size + multiple - 1) / multiple * multiple;
    if (padded == size) return t;
    std::vector<int64_t> sizes = t.sizes().vec();
    sizes[dim] = padded;
    const int64_t rows = dim == 0 ? 1 : t.numel() / std::max<int64_t>(size, 1), cols = dim == 0 ? t.numel() : size;
    if (cols == 0 || (dim == 0 ? cols / size * padded : padded) > INT32_MAX) {          // (no elements, or past the kernel's 32-bit widths)
        std::vector<int64_t> pad(2 * (t.dim() - dim), 0);
        pad.back() = padded - size;
        return at::constant_pad_nd(t, pad);
    }
    return copy_columns(t.contiguous(), rows, cols, sizes, dim == 0 ? cols / size * padded : padded, stream);
}

// What a kernel would otherwise find out by reading past a buffer or on another device.
void require_map(const Tensor& nmap, int64_t v) {
    if (nmap.dim() != 2 || nmap.size(1) != v)
        throw py::value_error("a neighbor cache of " + std::to_string(nmap.dim() == 2 ? nmap.size(1) : 0) + " kernel positions for a weight of " + std::to_string(v));
}
void require_on(const at::Device& dev, const Tensor& t, const char* what) {
    if (t.defined() && t.device() != dev) throw py::value_error(std::string(what) + " is on " + t.device().str() + ", the features on " + dev.str());
}

struct Product {
    Tensor out, mask;
    Tensor src;         // the rows as they were multiplied, where they had to be filled up to whole 16-byte pieces
};

// mode 0: out = conv(src) with weight [Co, V, Ci] (+ bias), mode 1: input gradient from src = grad_output through the same
// map with the offsets mirrored, mode 2: through a map of its own, offsets as they are.  One row per row of the cache's
// neighbor_map.  masked: mask-sorted schedule (else natural row order, all offsets per tile).  want_mask: also one bit per
// output, "greater than zero", where the kernels can (ReLU, 16-bit type, a multiple of 8 columns).  panel: the weight
// packed already, or undefined; owner: the tensor that a packed weight is kept with (null: none is kept).  Both only spare the packing of the
// kernels that read panels.
// Which kernel runs follows from shape, type and the plan that a narrow layer's cache has earned, never from whether gradients are recorded,
// a ReLU is asked for or its mask wanted: a recomputed pass, a fused and a composed ReLU, training and inference add in the same order and
// agree bit for bit.
Product gather_product(Tensor src, Tensor weight, Tensor bias, const Cache& c, int mode, bool allow_splitk, bool masked, int activation,
                       bool want_mask, const Tensor& panel_given, int64_t stream, py::handle owner = {}) {
    const at::Device dev = src.device();
    const c10::DeviceGuard guard(dev);
    const int code = dtype_code(src);
    if (weight.scalar_type() != src.scalar_type() || (bias.defined() && bias.scalar_type() != src.scalar_type()))
        throw py::type_error("features, weight and bias must share one dtype");
    const int es = (int)src.element_size(), v = (int)weight.size(1);
    const Tensor nmap = c.need("neighbor_map");
    require_map(nmap, v);
    require_on(dev, nmap, "the neighbor cache");
    require_on(dev, weight, "the weight");
    require_on(dev, bias, "the bias");
    const int64_t n = nmap.size(0), n_src = src.size(0);
    int cols = (int)weight.size(mode == 0 ? 0 : 2);
    if (bias.defined() && bias.numel() != cols)
        throw py::value_error("a bias of " + std::to_string(bias.numel()) + " values for " + std::to_string(cols) + " output channels");
    Product p;
    if (n_src == 0) {                       // nothing to gather: the bias alone
        p.out = at::zeros({n, cols}, src.options());
        if (bias.defined()) p.out = p.out + bias;
        if (activation == FGX_ACT_RELU) p.out = at::relu(p.out);
        return p;
    }
    const int align = 16 / es;
    if (weight.size(mode == 0 ? 2 : 0) % align) {       // rows must be whole 16-byte pieces
        owner = {};                                     // (a padded copy is made per call: nothing to keep a panel by)
        src = pad_to(src, 1, align, stream);
        weight = pad_to(weight, mode == 0 ? 2 : 0, align, stream);
        p.src = src;
    }
    src = src.contiguous();
    weight = weight.contiguous();
    if (bias.defined()) bias = bias.contiguous();
    int co = (int)weight.size(0), ci = (int)weight.size(2);
    const int k = mode == 0 ? ci : co;
    const int64_t row_bytes = (int64_t)k * es;
    const int pass = mode == 0 ? 0 : 1;
    // (these two kernels' outputs are whole 16-byte pieces: a ragged row is multiplied as one and cut)
    const int whole = es == 2 && schedules_are_ours() ? whole_columns(cols, n) : cols;
    // a network's first layers: all offsets of a row in one product, no row order or tile tables
    const bool stem = n > 0 && L.fgx_conv_gemm_stem_pays(code, mode, (size_t)n, k, whole, v) && schedules_are_ours() &&
                      aligned(src) && aligned(weight) && aligned(nmap);
    // Up to 32 channels on both sides: the resident-row kernel where it runs at once or the cache has earned its plan (38 720 voxels, 8 ->
    // 32 channels: 0.014 ms, 0.010 without; 98 408 voxels 0.015 and 0.016, 427 872 voxels 0.033 and 0.046, 16 -> 32 0.034 and 0.087).
    const bool narrow = n > 0 && narrow_shape(c, es, k, whole, v, n) &&
                        impl_function("_narrow_applies")(c.obj, src, k, whole, v, n, n_src,
                                                         python_schedule(pass, src, n, mode == 0 ? ci : whole, mode == 0 ? whole : co, v)).cast<bool>();
    const int cut = whole != cols && (stem || narrow) ? cols : 0;
    if (cut) {
        owner = {};
        weight = pad_to(weight, mode == 0 ? 0 : 2, align, stream);
        if (bias.defined()) bias = pad_to(bias, 0, align, stream);
        want_mask = false;                              // (one bit per output of the rows as they are)
        (mode == 0 ? co : ci) = cols = whole;
    }
    auto cut_back = [&] {
        if (cut) p.out = copy_columns(p.out, n, cols, {n, cut}, cut, stream);
    };
    if (stem && !narrow) {
        const char* name = mode == 0 ? "gather_gemm_fwd" : "gather_gemm_dgrad";
        p.out = make({n, cols}, src.scalar_type(), dev);
        if (want_mask && activation == FGX_ACT_RELU) p.mask = make({n * cols / 8}, at::kByte, dev);
        mark(name, "start");
        check(L.fgx_conv_gemm_stem(code, mode, ptr(src), ptr(weight), ptr(bias), ptr<uint32_t>(nmap), (size_t)n, ci, co, v, activation, ptr(p.out),
                                   ptr<uint8_t>(p.mask), as_stream(stream)));
        mark(name, "stop");
        cut_back();
        return p;
    }
    // few voxels under a small weight: one launch
    if (mode == 0 && masked && allow_splitk && !narrow && few_pays(code, n, ci, co, v) &&
        schedules_are_ours() && aligned(src) && aligned(weight)) {
        p.out = make({n, cols}, src.scalar_type(), dev);
        if (want_mask && activation == FGX_ACT_RELU && cols % 8 == 0) p.mask = make({n * cols / 8}, at::kByte, dev);
        mark("gather_gemm_fwd", "start");
        check(L.fgx_conv_gemm_few_mask(code, ptr(src), ptr(weight), ptr(bias), ptr<uint32_t>(nmap), (size_t)n, ci, co, v, activation, ptr(p.out),
                                       ptr<uint8_t>(p.mask), as_stream(stream)));
        mark("gather_gemm_fwd", "stop");
        return p;
    }
    // few voxels under a wide weight: the pairs' products and their sums, from a plan of the map that every layer on it shares
    if (masked && allow_splitk && n > 0 && !narrow && L.fgx_conv_gemm_pairs_pays(code, mode, (size_t)n, ci, co, v) &&
        schedules_are_ours() && aligned(src) && aligned(weight) && (double)n_src * row_bytes <= (double)0xFF000000u) {
        Tensor plan;
        if (!c.tensor("_pair_plan", &plan)) {
            plan = make({(int64_t)L.fgx_pair_plan_words((size_t)n, v)}, at::kUInt32, dev);
            check(L.fgx_pair_plan(ptr<uint32_t>(nmap), (size_t)n, v, ptr<uint32_t>(plan), as_stream(stream)));
            c.set("_pair_plan", plan);
        }
        Tensor scratch = workspace(L.fgx_conv_gemm_pairs_scratch_bytes((size_t)n, cols, v), dev);
        p.out = make({n, cols}, src.scalar_type(), dev);
        if (want_mask && activation == FGX_ACT_RELU && es == 2) p.mask = make({n * cols / 8}, at::kByte, dev);
        const char* name = mode == 0 ? "gather_gemm_fwd" : "gather_gemm_dgrad";
        mark(name, "start");
        check(L.fgx_conv_gemm_pairs(code, mode, ptr(src), ptr(weight), ptr(bias), ptr<uint32_t>(plan), (size_t)n, (size_t)n_src, ci, co, v, ptr(scratch),
                                    activation, ptr(p.out), ptr<uint8_t>(p.mask), as_stream(stream)));
        mark(name, "stop");
        return p;
    }
    if (masked && !narrow && !(c.has("gray_code") && c.has("sorted_idx"))) {
        if (c.has("_order_left_out")) cache_post(c, true, false);
        else {
            const py::tuple made = impl_function("_codes_and_order")(nmap, py::none(), py::none());
            c.set("gray_code", made[0].cast<Tensor>());
            c.set("sorted_idx", made[2].cast<Tensor>());
        }
    }
    Sched s = schedule(pass, src, n, ci, co, v);
    bool own_order = false;
    if (masked && !narrow && row_bytes <= module_int(g_impl, "LOCALITY_MAX_ROW_BYTES") && (c.has("_tile_order") || n >= module_int(g_impl, "LOCALITY_MIN_ROWS")) &&
        impl_function("_locality_applies")(c.obj, n, row_bytes).cast<bool>()) {
        c.tables_by([&] { return c.obj.attr("_ensure_tile_order")(); });
        own_order = c.has("_tile_order");
    }
    if (n == 0) {
        p.out = make({n, cols}, src.scalar_type(), dev);
        return p;
    }
    // the streaming kernel addresses its operands with 32-bit byte offsets
    const double most = (double)0xFF000000u;
    const bool streams = s.stream && (double)n_src * row_bytes <= most && (double)n * 8 <= most && (double)n * 27 * 4 * 2 <= most;
    Tensor panel = panel_given;
    if (s.stream && !streams && !(s.tile_rows == 256 && s.tile_cols == 128)) {      // a streaming tile that the tiled kernel, which addresses more, does not have
        s = Sched{128, cols > 64 ? 128 : cols > 32 ? 64 : 32, 64, 1, 0, 0};
        panel = Tensor();                               // (packed for the other tile)
        owner = {};
    }
    if (!panel.defined() && owner)
        panel = impl_function("_weight_panel")(owner, weight, code, mode, python_schedule(pass, src, n, ci, co, v), py::cast(src).attr("device")).cast<Tensor>();
    // the tiled kernel reads the weight itself where it can
    const bool direct = !panel.defined() && !narrow && !streams && aligned(weight) && L.fgx_conv_gather_gemm_weight_pays(code, mode, ci, co, v);
    if (!direct && !panel.defined()) {
        panel = workspace(L.fgx_weight_panel_bytes(code, mode, ci, co, v, s.slab_bytes, s.tile_cols), dev);
        check(L.fgx_pack_weight(code, mode, ptr(weight), ci, co, v, s.slab_bytes, s.tile_cols, ptr(panel), as_stream(stream)));
    }
    c.wait_for_tables();
    if (narrow) {
        const py::tuple got = c.tables_by([&] {
            return py::tuple(impl_function("_narrow_gemm")(src, panel, bias.defined() ? py::cast(bias) : py::none(), c.obj, mode, k, cols, v, activation, want_mask));
        });
        p.out = got[0].cast<Tensor>();
        if (!got[1].is_none()) p.mask = got[1].cast<Tensor>();
        cut_back();
        return p;
    }
    p.out = make({n, cols}, src.scalar_type(), dev);
    if (want_mask && activation == FGX_ACT_RELU && es == 2 && cols % 8 == 0) p.mask = make({n * cols / 8}, at::kByte, dev);
    const void* b = ptr(bias);
    const char* name = mode == 0 ? "gather_gemm_fwd" : "gather_gemm_dgrad";
    if (streams) {
        int groups = 0;
        check(L.fgx_conv_gather_gemm_stream_groups(code, cols, s.tile_rows, s.tile_cols, s.slab_bytes, &groups));
        Tensor item_at;
        const Tiles t = gather_plan(c, s.tile_rows, own_order, !masked, ceil_div(cols, s.tile_cols), groups, ceil_div(row_bytes, s.slab_bytes), &item_at,
                                    stream);
        mark(name, "start");
        check(L.fgx_conv_gather_gemm_stream_act_mask(code, ptr(src), ptr(panel), b, ptr<int64_t>(t.order), ptr<int32_t>(t.code),
                                                     ptr<int32_t>(t.plan_seg), ptr<uint32_t>(t.plan_idx), ptr<uint32_t>(t.plan_band),
                                                     (size_t)t.plan_idx.size(0), (size_t)n, (size_t)n_src, k, cols, v, s.tile_rows, s.tile_cols,
                                                     s.slab_bytes, ptr<uint32_t>(item_at), groups, activation, ptr(p.out), ptr<uint8_t>(p.mask),
                                                     as_stream(stream)));
    } else {
        const int splitk = allow_splitk ? s.splitk : 1;
        Tiles t;
        if (masked) {
            tile_codes(c, s.tile_rows, own_order, stream, &t, false);
        } else {
            const py::tuple oc = c.tables_by([&] { return py::tuple(c.obj.attr("_dense_tile_tables")(s.tile_rows)); });
            t.order = oc[0].cast<Tensor>();
            t.code = oc[1].cast<Tensor>();
        }
        Tensor scratch;
        if (splitk > 1) scratch = workspace(L.fgx_conv_scratch_bytes((size_t)n, cols, splitk), dev);
        mark(name, "start");
        if (direct)
            check(L.fgx_conv_gather_gemm_weight(code, mode, ptr(src), ptr(weight), b, ptr<uint32_t>(nmap), ptr<int64_t>(t.order), ptr<int32_t>(t.code),
                                                (size_t)n, ci, co, v, s.tile_rows, s.tile_cols, s.slab_bytes, splitk, ptr(scratch), activation,
                                                ptr(p.out), ptr<uint8_t>(p.mask), as_stream(stream)));
        else
            check(L.fgx_conv_gather_gemm_act_mask(code, ptr(src), ptr(panel), b, ptr<uint32_t>(nmap), ptr<int64_t>(t.order), ptr<int32_t>(t.code),
                                                  (size_t)n, k, cols, v, s.tile_rows, s.tile_cols, s.slab_bytes, splitk, ptr(scratch), activation,
                                                  ptr(p.out), ptr<uint8_t>(p.mask), as_stream(stream)));
    }
    mark(name, "stop");
    return p;
}

py::tuple gather_gemm(const Tensor& src, const Tensor& weight, const c10::optional<Tensor>& bias, py::object cache, int mode, bool allow_splitk,
                      bool masked, int activation, bool want_mask, const c10::optional<Tensor>& panel, py::object owner) {
    const Product p = gather_product(src, weight, bias.value_or(Tensor()), Cache(std::move(cache), stream_of(src)), mode, allow_splitk, masked, activation, want_mask,
                                     panel.value_or(Tensor()), stream_of(src), owner.is_none() ? py::handle() : owner);
    return py::make_tuple(p.out, p.mask.defined() ? py::cast(p.mask) : py::none());
}

// [V + 1] words of the segment table on the host
std::vector<uint32_t> seg_host(const Cache& c, int v) {
    PyObject* kept = c.find("_valid_signal_seg_host");
    py::sequence words = kept != nullptr ? py::reinterpret_borrow<py::sequence>(kept) : c.obj.attr("_seg_host")().cast<py::sequence>();
    if ((int)py::len(words) != v + 1) throw py::value_error("valid_signal_seg does not fit the pair lists (V + 1 entries, the last one their length)");
    std::vector<uint32_t> out((size_t)v + 1);
    for (int i = 0; i <= v; ++i) out[i] = words[i].cast<uint32_t>();
    return out;
}

Tensor wgrad_bounds(const Cache& c, const Tensor& sig_o, const std::vector<uint32_t>& seg, size_t n, int v, int block_rows, int64_t stream) {
    const std::string key = "_wgrad_bounds_" + std::to_string(block_rows);
    Tensor bounds;
    if (c.tensor(key, &bounds)) return bounds;
    const int64_t count = (int64_t)L.fgx_wgrad_block_bounds_count(n, v, block_rows);
    bounds = make({std::max<int64_t>(count, 1)}, at::kUInt32, sig_o.device());
    check(L.fgx_wgrad_block_bounds(ptr<uint32_t>(sig_o), seg.data(), n, v, block_rows, ptr<uint32_t>(bounds), as_stream(stream)));
    c.set(key, bounds);
    return bounds;
}

Tensor wgrad_item_lists(const Cache& c, const Tensor& bounds, size_t n, int v, int ci, int co, const Sched& s, bool only_if_they_pay, int64_t stream) {
    const std::string key = "_wgrad_lists_" + std::to_string(s.block_rows) + "_" + std::to_string(s.tile_rows) + "_" + std::to_string(s.tile_cols) +
                            "_" + std::to_string(ci) + "_" + std::to_string(co);
    Tensor lists;
    if (PyObject* kept = c.find(key)) {
        if (THPVariable_Check(kept)) lists = THPVariable_Unpack(kept);
        return lists;                                   // (None: the library has none for the shape)
    }
    const size_t words = L.fgx_wgrad_item_lists_count(n, v, ci, co, s.tile_rows, s.tile_cols, s.block_rows);
    // with no more items than workgroups there is nothing to even out, and the fixed interleave hands out one item each
    // (3 716 voxels, 64 channels: 108 items; making their lists took 18 us beside a weight gradient of 12)
    const size_t items = (size_t)v * ceil_div(co, s.tile_rows) * ceil_div(ci, s.tile_cols) * (size_t)ceil_div((int64_t)n, s.block_rows);
    if (only_if_they_pay && words > 0 && items <= words - 4 - items) return lists;
    if (words > 0) {
        lists = make({(int64_t)words}, at::kUInt32, bounds.device());
        check(L.fgx_wgrad_item_lists(ptr<uint32_t>(bounds), n, v, ci, co, s.tile_rows, s.tile_cols, s.block_rows, ptr<uint32_t>(lists), as_stream(stream)));
        c.set(key, lists);
    } else {
        c.set(key, py::none());
    }
    return lists;
}

bool sweep_fits(int64_t n, int64_t n_in, int64_t ci, int64_t co, int es, int64_t pairs) {
    return pairs > 0 && L.fgx_wgrad_sweep_fits((size_t)n, (size_t)n_in, (int)ci, (int)co, es, (size_t)pairs);
}

struct WeightGrads {
    Tensor weight, bias;
};

// [Co, V, Ci] weight gradient (and with with_bias the bias gradient) from the cache's pair lists: grad has one row per row of
// the cache's map, feats one per row the map points at.  bias_offset names an offset whose pairs hold every row of grad exactly
// once (-1: none), which lets the streaming kernel sum the rows it loads anyway.  true_ci, true_co: the channels, where the rows come filled up.
WeightGrads weight_grads(Tensor grad, Tensor feats, const Cache& c, int v, bool with_bias, int bias_offset, int64_t stream, int64_t true_ci = -1,
                         int64_t true_co = -1) {
    const at::Device dev = feats.device();
    const c10::DeviceGuard guard(dev);
    const int code = dtype_code(feats);
    {
        const Tensor nmap = c.need("neighbor_map");
        require_map(nmap, v);
        require_on(dev, nmap, "the neighbor cache");
        require_on(dev, grad, "the upstream gradient");
        if (grad.size(0) != nmap.size(0))
            throw py::value_error(std::to_string(grad.size(0)) + " gradient rows for a neighbor cache of " + std::to_string(nmap.size(0)) + " rows");
    }
    const int64_t n = grad.size(0), n_in = feats.size(0);
    if (true_ci < 0) true_ci = feats.size(1);
    if (true_co < 0) true_co = grad.size(1);
    const int es = (int)feats.element_size(), align = 16 / es;
    feats = pad_to(feats, 1, align, stream).contiguous();
    grad = pad_to(grad, 1, align, stream).contiguous();
    const int ci = (int)feats.size(1), co = (int)grad.size(1);
    WeightGrads w;
    if (n > 0 && narrow_shape(c, es, ci, co, v, n) && impl_function("_narrow_wgrad_applies")(c.obj, feats, ci, co, v, n, n_in).cast<bool>()) {
        const py::tuple got = c.tables_by([&] { return py::tuple(impl_function("_narrow_wgrad")(grad, feats, c.obj, v, with_bias)); });
        w.weight = got[0].cast<Tensor>();
        if (with_bias) w.bias = got[1].cast<Tensor>();
    } else if (L.fgx_wgrad_stem_pays(code, (size_t)n, ci, co, v) && n_in > 0 && schedules_are_ours() && aligned(feats) && aligned(grad) &&
               aligned(c.need("neighbor_map"))) {
        const Tensor nmap = c.need("neighbor_map");
        Tensor scratch = workspace(L.fgx_wgrad_stem_scratch_bytes((size_t)n, ci, co), dev);
        w.weight = make({co, v, true_ci}, feats.scalar_type(), dev);
        if (with_bias) w.bias = make({co}, feats.scalar_type(), dev);
        mark("wgrad", "start");
        check(L.fgx_conv_wgrad_stem_cut(code, ptr(grad), ptr(feats), ptr<uint32_t>(nmap), (size_t)n, ci, (int)true_ci, co, v, ptr(scratch), ptr(w.weight),
                                        ptr(w.bias), as_stream(stream)));
        mark("wgrad", "stop");
    } else {
        if (!(c.has("valid_signal_seg") && (c.has("valid_signal_i") || c.has("_pending_pairs")))) {
            refuse_lists_in_capture(stream);
            c.tables_by([&] { return c.obj.attr("_ensure_pairs")(); });
        }
        const Tensor sig_i = c.need("valid_signal_i"), sig_o = c.need("valid_signal_o");
        const std::vector<uint32_t> seg = seg_host(c, v);
        c.wait_for_tables();
        const int64_t pairs = seg[v];
        if (pairs > std::min(sig_i.numel(), sig_o.numel()))
            throw py::value_error("valid_signal_seg does not fit the pair lists (V + 1 entries, the last one their length)");
        Sched s;
        if (schedules_are_ours()) {
            fgx_schedule got;
            check(L.fgx_wgrad_schedule(code, (size_t)n, (size_t)n_in, (uint32_t)pairs, ci, co, v, &got));
            memcpy(&s, &got, sizeof(s));
        } else {                            // a forced one, within what its kernel takes
            s = schedule(2, feats, n, ci, co, v);
            if (s.stream == 1 && code == FGX_F32 && s.tile_rows == s.tile_cols &&
                L.fgx_conv_wgrad_split_scratch_bytes((size_t)n, (size_t)n_in, (uint32_t)pairs, v, ci, co, s.tile_rows, s.block_rows) > 0)
                s.stream = 3;
            if (s.stream == 2 && !sweep_fits(n, n_in, ci, co, es, pairs)) {
                s.stream = 1;
                s.block_rows = 12288;
            }
        }
        w.weight = make({co, v, ci}, feats.scalar_type(), dev);
        if (with_bias) w.bias = make({co}, feats.scalar_type(), dev);
        if (s.stream == 2) {
            const std::string key = "_wgrad_sweep_plan_" + std::to_string(s.block_rows);
            Tensor plan;
            if (!c.tensor(key, &plan)) {
                plan = workspace(L.fgx_wgrad_sweep_plan_bytes((size_t)n, (size_t)pairs, v, s.block_rows), dev);
                check(L.fgx_wgrad_sweep_plan(ptr<uint32_t>(sig_o), seg.data(), (size_t)n, v, s.block_rows, ptr(plan), (size_t)plan.numel(),
                                             as_stream(stream)));
                c.set(key, plan);
            }
            Tensor scratch = workspace(L.fgx_wgrad_sweep_scratch_bytes(ci, co), dev);
            mark("wgrad", "start");
            check(L.fgx_conv_wgrad_sweep(code, ptr(grad), ptr(feats), ptr<uint32_t>(sig_i), ptr<uint32_t>(sig_o), seg.data(), ptr(plan), (size_t)n,
                                         (size_t)n_in, ci, co, v, s.tile_rows, s.block_rows, (int)module_int(g_impl, "WGRAD_SWEEP_LEAD"),
                                         (int)module_int(g_impl, "WGRAD_SWEEP_MAX_POLLS"), ptr(scratch), ptr(w.weight), ptr(w.bias), bias_offset,
                                         as_stream(stream)));
        } else {
            const Tensor bounds = wgrad_bounds(c, sig_o, seg, (size_t)n, v, s.block_rows, stream);
            Tensor lists;
            const size_t split = s.stream == 3 ? L.fgx_conv_wgrad_split_scratch_bytes((size_t)n, (size_t)n_in, (uint32_t)pairs, v, ci, co, s.tile_rows, s.block_rows) : 0;
            if (s.stream == 1 && code != FGX_F32 && PyObject_IsTrue(module_get(g_impl, "WGRAD_BALANCED_LISTS")))
                lists = wgrad_item_lists(c, bounds, (size_t)n, v, ci, co, s, true, stream);
            Tensor scratch = workspace(split ? split : L.fgx_wgrad_scratch_bytes((size_t)n, v, ci, co, s.block_rows), dev);
            mark("wgrad", "start");
            if (split)
                check(L.fgx_conv_wgrad_split(ptr(grad), ptr(feats), ptr<uint32_t>(sig_i), ptr<uint32_t>(sig_o), seg.data(), ptr<uint32_t>(bounds),
                                             (size_t)n, (size_t)n_in, ci, co, v, s.tile_rows, s.block_rows, ptr(scratch), ptr(w.weight), ptr(w.bias),
                                             as_stream(stream)));
            else
                check(L.fgx_conv_wgrad_lists(code, ptr(grad), ptr(feats), ptr<uint32_t>(sig_i), ptr<uint32_t>(sig_o), seg.data(), ptr<uint32_t>(bounds),
                                             ptr<uint32_t>(lists), (size_t)n, (size_t)n_in, ci, co, v, s.tile_rows, s.tile_cols, s.block_rows, s.stream,
                                             ptr(scratch), ptr(w.weight), ptr(w.bias), bias_offset, as_stream(stream)));
        }
        mark("wgrad", "stop");
    }
    if (ci != true_ci || co != true_co) {
        w.weight = w.weight.slice(0, 0, true_co).contiguous();              // (a view: whole rows)
        if (w.weight.numel() != true_co * v * true_ci) w.weight = copy_columns(w.weight, true_co * v, ci, {true_co, v, true_ci}, true_ci, stream);
        if (with_bias) w.bias = w.bias.slice(0, 0, true_co).contiguous();
    }
    return w;
}

py::tuple wgrad(const Tensor& grad, const Tensor& feats, py::object cache, int v, bool with_bias, int bias_offset) {
    const WeightGrads w = weight_grads(grad, feats, Cache(std::move(cache), stream_of(feats)), v, with_bias, bias_offset, stream_of(feats));
    return py::make_tuple(w.weight, w.bias.defined() ? py::cast(w.bias) : py::none());
}

Tensor relu_mask_apply(const Tensor& grad, const Tensor& mask, int64_t stream) {
    const c10::DeviceGuard guard(grad.device());
    const Tensor g = grad.contiguous();
    Tensor out = at::empty_like(g);
    check(L.fgx_relu_mask_apply(dtype_code(g), ptr(g), ptr<uint8_t>(mask), (size_t)g.numel(), ptr(out), as_stream(stream)));
    return out;
}

Tensor colsum(const Tensor& grad, int64_t stream) {
    const c10::DeviceGuard guard(grad.device());
    const int64_t n = grad.size(0), co = grad.size(1);
    Tensor out = make({co}, grad.scalar_type(), grad.device());
    Tensor scratch = workspace(L.fgx_colsum_scratch_bytes((size_t)n, (int)co), grad.device());
    check(L.fgx_colsum(dtype_code(grad), ptr(grad), (size_t)n, (int)co, ptr(scratch), ptr(out), as_stream(stream)));
    return out;
}

// ---- the differentiable operators --------------------------------------------------------------------------------------
// What one call of an operator is: kept by its node for the backward pass.
struct Call {
    bool generic = false;               // sparse_conv3d: an input gradient through a map of its own
    bool masked = true, splitk = true;  // the algorithm's schedule
};

// A Python object held where the interpreter lock may not be.
struct Held {
    PyObject* obj = nullptr;
    ~Held() { drop(); }
    void take(py::handle h) {
        obj = h.ptr();
        Py_INCREF(obj);
    }
    void drop() {
        if (obj != nullptr && Py_IsInitialized()) {
            const py::gil_scoped_acquire gil;
            Py_CLEAR(obj);
        }
    }
};

using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// Features with their rows filled up are kept to the backward pass, beside the features themselves, up to this size a layer, a thousandth of the card's memory:
// filling them up again costs 3 to 4 % of a training pass over many rows (166 232 voxels, 82 channels, four layers 1 230 -> 1 274 us; 406 920, 27
// channels, three 490 -> 513; level up to 82 400), keeping them doubles what ragged layers hold between their passes (the four layers 109 -> 226 MB,
// at the peak 295 -> 328).
constexpr int64_t kFilledKeptBytes = 256 << 20;

struct ConvBackward : public torch::autograd::Node {
    Call call;
    Held cache;
    SavedVariable feats, weight, bias, output;      // (the bias only to refuse one that was changed in place)
    SavedVariable mask;                 // the ReLU's derivative, one bit per output
    Tensor filled;                      // feats with its rows filled up, as the forward pass had them (undefined: the backward pass fills its own)
    bool relu = false, has_bias = false, has_mask = false;

    std::string name() const override { return call.generic ? "SparseConv3dBackward" : "SubMConv3dBackward"; }
    void release_variables() override {
        feats.reset_data();
        weight.reset_data();
        bias.reset_data();
        output.reset_data();
        mask.reset_data();
        filled.reset();
    }

    variable_list apply(variable_list&& grads) override {
        try {
            return gradients(std::move(grads));
        } catch (py::error_already_set& e) {        // keep the Python error's type on its way through the engine's thread
            const py::gil_scoped_acquire gil;
            e.restore();
            throw_persistent();
        } catch (py::builtin_exception& e) {        // (py::value_error and its like, which become one only in pybind's hands)
            const py::gil_scoped_acquire gil;
            e.set_error();
            throw_persistent();
        }
    }
    [[noreturn]] static void throw_persistent() {
        python_error err;
        err.persist();
        throw err;
    }

    variable_list gradients(variable_list&& grads) {
        variable_list result(has_bias ? 3 : 2);
        if (!grads[0].defined()) return result;
        const bool need_f = task_should_compute_output(0), need_w = task_should_compute_output(1);
        const bool need_b = has_bias && task_should_compute_output(2);
        // (before anything else: a hook of the saved tensors may run the caller's code here)
        const Tensor f = feats.unpack(), w = weight.unpack(), m = has_mask ? mask.unpack() : Tensor();
        const Tensor y = relu && !has_mask ? output.unpack(shared_from_this()) : Tensor();
        if (has_bias) (void)bias.unpack();
        for (const Tensor* t : {&f, &w, &m, &y})             // (... and may leave one where the kernels cannot read it)
            if (t->defined() && t->device() != grads[0].device())
                throw py::value_error("a saved tensor of " + name() + " is on " + t->device().str() + ", the gradient on " + grads[0].device().str());
        const at::NoGradGuard no_grad;
        const py::gil_scoped_acquire gil;
        const int64_t stream = stream_of(f);
        const Cache c(py::reinterpret_borrow<py::object>(cache.obj), stream);
        // rows filled up once for both products
        Tensor grad = grads[0];
        const int64_t align = 16 / (int64_t)grad.element_size(), rows = grad.size(0), filled_co = (grad.size(1) + align - 1) / align * align;
        if (has_mask) {
            grad = relu_mask_apply(grad, m, stream);
        } else if (relu && grad.numel() > 0 && y.scalar_type() == grad.scalar_type() && y.sizes() == grad.sizes()) {
            const Tensor g = grad.contiguous(), h = y.contiguous();
            grad = make({rows, filled_co}, g.scalar_type(), g.device());
            check(L.fgx_relu_columns(dtype_code(g), ptr(g), ptr(h), (size_t)rows, (int)g.size(1), ptr(grad), (int)filled_co, as_stream(stream)));
        } else if (relu) {
            grad = at::where(y.gt(0), grad, at::zeros({}, grad.options()));
        }
        grad = pad_to(grad.contiguous(), 1, align, stream);
        const int64_t co = w.size(0), kw = w.size(1), kh = w.size(2), kd = w.size(3), ci = w.size(4), v = kw * kh * kd;
        if (need_f) {
            const Tensor wv = w.reshape({co, v, ci});
            if (call.generic) {
                const Cache view(c.obj.attr("_bwd_view")(), stream);
                // mask-sorted walk only where the cache carries the backward order
                result[0] = gather_product(grad, wv, Tensor(), view, 2, call.splitk, call.masked && view.has("sorted_idx"), FGX_ACT_NONE, false, Tensor(),
                                           stream).out;
            } else {
                result[0] = gather_product(grad, wv, Tensor(), c, 1, call.splitk, call.masked, FGX_ACT_NONE, false, Tensor(), stream).out;
            }
        }
        if (need_w) {
            // odd submanifold kernel: the centre offset pairs every voxel with itself, so the bias gradient rides along
            const bool odd = kw % 2 && kh % 2 && kd % 2 && !call.generic;
            const int centre = odd && PyObject_IsTrue(module_get(g_spconv, "FUSE_DBIAS")) ? (int)(v / 2) : -1;
            const bool with_bias = need_b && !call.generic;
            WeightGrads g = weight_grads(grad, filled.defined() ? filled : f, c, (int)v, with_bias, with_bias ? centre : -1, stream, ci, co);
            result[1] = g.weight.reshape({co, kw, kh, kd, ci});
            if (with_bias) result[2] = g.bias;
        }
        if (need_b && !result[2].defined()) result[2] = colsum(grad, stream).slice(0, 0, co);
        return result;
    }
};

void require(bool ok, const std::string& what) {
    if (ok) return;
    PyErr_SetString(PyExc_AssertionError, what.c_str());
    throw py::error_already_set();
}

// One layer: its output, with a node behind it when gradients are recorded.  cache: the neighbor cache of its coordinates.
Tensor convolve(const Tensor& feats, py::object cache_obj, const Tensor& weight, const c10::optional<Tensor>& bias_opt, bool relu, bool generic,
                bool masked, bool splitk) {
    const Tensor bias = bias_opt.value_or(Tensor());
    const bool has_bias = bias.defined();
    const bool record = at::GradMode::is_enabled() && (feats.requires_grad() || weight.requires_grad() || (has_bias && bias.requires_grad()));
    require(weight.dim() == 5 && feats.dim() == 2, "features are [N, C], weights [Co, Kw, Kh, Kd, Ci]");
    const int64_t co = weight.size(0), v = weight.size(1) * weight.size(2) * weight.size(3), ci = weight.size(4);
    require(feats.size(1) == ci, "Input channels (" + std::to_string(feats.size(1)) + ") should match weight channels (" + std::to_string(ci) + ")");
    require(feats.is_contiguous(), "Input features should be contiguous");
    const Cache c(std::move(cache_obj), stream_of(feats));
    int64_t expected = c.need("neighbor_map").size(0);
    if (generic) {                      // rows of the input the maps were made for (absent on a hand-made cache)
        expected = feats.size(0);
        Tensor bwd;
        if (PyObject* m = c.find("_n_in")) {
            if (m != Py_None) expected = PyLong_AsLongLong(m);
        } else if (c.tensor("neighbor_map_bwd", &bwd)) {
            expected = bwd.size(0);
        }
    }
    require(feats.size(0) == expected, std::to_string(feats.size(0)) + " feature rows for a neighbor cache of " + std::to_string(expected) + " voxels");
    // lists that the layer the cache was built for does not read and this one's weight gradient will: on their way from here on, so that
    // the backward pass does not wait for their length
    if (record && weight.requires_grad() && c.has("_lists_left_out") && !capturing(stream_of(feats))) {
        const Layer l{dtype_code(feats), ci, co, true, feats.requires_grad(), true, splitk};
        if (layer_needs(l, feats.size(0), (int)v, c.has("_cell_walk")).lists) cache_post(c, false, true);
    }
    const bool bits = relu && record && PyObject_IsTrue(module_get(g_spconv, "RELU_BIT_MASK"));
    Product p;
    {
        const at::NoGradGuard no_grad;
        p = gather_product(feats, weight.reshape({co, v, ci}), bias, c, 0, splitk, masked, relu ? FGX_ACT_RELU : FGX_ACT_NONE, bits, Tensor(),
                           stream_of(feats));
    }
    if (!record) return p.out;
    // (deleteNode: a long chain of layers is taken down without a stack frame per layer)
    const std::shared_ptr<ConvBackward> node(new ConvBackward(), torch::autograd::deleteNode);
    node->set_next_edges(has_bias ? torch::autograd::collect_next_edges(feats, weight, bias) : torch::autograd::collect_next_edges(feats, weight));
    node->call.generic = generic;
    node->call.masked = masked;
    node->call.splitk = splitk;
    node->cache.take(c.obj);
    node->relu = relu;
    node->has_bias = has_bias;
    node->feats = SavedVariable(feats, false);
    node->weight = SavedVariable(weight, false);
    if (has_bias) node->bias = SavedVariable(bias, false);
    // (hooks of the saved tensors may want nothing left on the device)
    if (p.src.defined() && weight.requires_grad() && (int64_t)p.src.nbytes() <= kFilledKeptBytes && !at::SavedTensorDefaultHooks::get_hooks().has_value())
        node->filled = p.src;
    node->has_mask = p.mask.defined();
    if (node->has_mask) node->mask = SavedVariable(p.mask, false);
    torch::autograd::set_history(p.out, node);
    if (relu && !p.mask.defined()) node->output = SavedVariable(p.out, true);
    return p.out;
}

// ---- curve codes -----------------------------------------------------------------------------------------------------
Tensor encode(const Tensor& coords, int mode, int bits, int code_bits) {
    const c10::DeviceGuard guard(coords.device());
    const Tensor c = coords.contiguous();
    Tensor codes = make({c.size(0)}, code_bits == 32 ? at::kInt : at::kLong, c.device());
    check(L.fgx_serialize_encode(mode, ptr<int32_t>(c), (size_t)c.size(0), bits, code_bits, ptr(codes), as_stream(stream_of(c))));
    return codes;
}

Tensor decode(const Tensor& codes, int mode, int bits, int code_bits) {
    const c10::DeviceGuard guard(codes.device());
    const Tensor c = codes.contiguous();
    Tensor coords = make({c.size(0), 4}, at::kInt, c.device());
    check(L.fgx_serialize_decode(mode, ptr(c), (size_t)c.size(0), bits, code_bits, ptr<int32_t>(coords), as_stream(stream_of(c))));
    return coords;
}

// ---- the Python methods of the cache that make tables by themselves ----------------------------------------------------
Cache on_its_stream(py::object cache) {
    const int64_t stream = stream_of(cache.attr("neighbor_map").cast<Tensor>());
    return Cache(std::move(cache), stream);
}

// The mask order of a cache that was built without it (a recorded one during a capture, which is not the cache's).
Tensor py_cache_order(py::object cache_obj) {
    const Cache c = on_its_stream(std::move(cache_obj));
    Tensor order;
    if (!c.tensor("sorted_idx", &order)) cache_post(c, true, false);
    return c.need("sorted_idx");
}

py::tuple py_tile_codes(py::object cache_obj, int block, bool own_order) {
    const Cache c = on_its_stream(std::move(cache_obj));
    Tiles t;
    const Tensor nmap = c.need("neighbor_map");
    const c10::DeviceGuard guard(nmap.device());
    tile_codes(c, block, own_order, stream_of(nmap), &t, false);
    return py::make_tuple(t.order, t.code);
}

py::tuple py_gather_plan(py::object cache_obj, int block, bool own_order, bool dense) {
    const Cache c = on_its_stream(std::move(cache_obj));
    const Tensor nmap = c.need("neighbor_map");
    const c10::DeviceGuard guard(nmap.device());
    const Tiles t = gather_plan(c, block, own_order, dense, 0, 0, 0, nullptr, stream_of(nmap));
    return py::make_tuple(t.order, t.code, t.plan_seg, t.plan_idx, t.plan_band, t.plan_key);
}

py::object py_item_order(py::object cache_obj, const std::string& plan_key, const Tensor& code, int col_tiles, int groups, int slabs) {
    const Cache c = on_its_stream(std::move(cache_obj));
    const c10::DeviceGuard guard(code.device());
    const Tensor t = item_order(c, plan_key, code, col_tiles, groups, slabs, stream_of(code));
    return t.defined() ? py::cast(t) : py::none();
}

py::object py_wgrad_bounds(py::object cache_obj, int block_rows) {
    const Cache c = on_its_stream(std::move(cache_obj));
    const Tensor nmap = c.need("neighbor_map"), sig_o = c.need("valid_signal_o");
    const c10::DeviceGuard guard(nmap.device());
    const int v = (int)nmap.size(1);
    return py::cast(wgrad_bounds(c, sig_o, seg_host(c, v), (size_t)nmap.size(0), v, block_rows, stream_of(nmap)));
}

py::object py_wgrad_item_lists(py::object cache_obj, int block_rows, int tile_rows, int tile_cols, int ci, int co) {
    const Tensor bounds = py_wgrad_bounds(cache_obj, block_rows).cast<Tensor>();
    const Cache c = on_its_stream(std::move(cache_obj));
    const Tensor nmap = c.need("neighbor_map");
    const c10::DeviceGuard guard(nmap.device());
    const Sched s{tile_rows, tile_cols, 0, 1, block_rows, 1};
    const Tensor t = wgrad_item_lists(c, bounds, (size_t)nmap.size(0), (int)nmap.size(1), ci, co, s, false, stream_of(nmap));
    return t.defined() ? py::cast(t) : py::none();
}

}  // namespace

PYBIND11_MODULE(fgx_host, m) {
    py::class_<SegHost>(m, "SegHost").def("synchronize", &SegHost::synchronize).def("tolist", &SegHost::tolist);
    m.def("bind", &bind);
    m.def("subm_cache", &subm_cache);
    m.def("cache_order", &py_cache_order);
    m.def("cache_lists", [](py::object cache) { cache_post(on_its_stream(std::move(cache)), false, true); });
    m.def("spconv_cache", &spconv_cache);
    m.def("out_coords", &out_coords);
    m.def("convolve", &convolve);
    m.def("gather_gemm", &gather_gemm, py::arg("src"), py::arg("weight"), py::arg("bias"), py::arg("cache"), py::arg("mode"), py::arg("allow_splitk"),
          py::arg("masked"), py::arg("activation"), py::arg("want_mask"), py::arg("panel") = py::none(), py::arg("owner") = py::none());
    m.def("wgrad", &wgrad);
    m.def("sweep_fits", &sweep_fits);
    m.def("relu_mask_apply", [](const Tensor& grad, const Tensor& mask) { return relu_mask_apply(grad, mask, stream_of(grad)); });
    m.def("colsum", [](const Tensor& grad) { return colsum(grad, stream_of(grad)); });
    m.def("encode", &encode);
    m.def("decode", &decode);
    m.def("tile_codes", &py_tile_codes);
    m.def("gather_plan", &py_gather_plan);
    m.def("item_order", &py_item_order);
    m.def("wgrad_bounds", &py_wgrad_bounds);
    m.def("wgrad_item_lists", &py_wgrad_item_lists);
}

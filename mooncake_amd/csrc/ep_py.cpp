// mooncake_amd._ep: the compiled Python module of this library, a drop-in for the
// reference's pybind11 module `mooncake._ep` on the low-latency dispatch / combine
// path (mooncake-ep/src/ep_py.cpp:14-46): get_ep_buffer_size_hint, MAX_QP_COUNT,
// EventHandle, Buffer with the bound names and argument order of the reference, and
// _benchmark_legacy_buffer with its three structs
// (mooncake-ep/benchmarks/legacy_buffer_perf.cpp:151-199).  Everything goes through
// the C ABI of include/mooncake_ep_hip.h; in what the reference binds no torch type
// appears here either - device addresses and streams are integers, as there.
//
// Buffer.dispatch_tensors and combine_tensors are the exception: the reference wrapper's
// checks, its outputs and the call itself in one native step, for the Python `Buffer`
// above (a rank's dispatch took 4.1 us of host time through Python and a combine 5.2,
// nearly all of it tensor attributes, torch.empty and the pool's look-up).  So are
// World.dispatch_stacked, combine_stacked and cast_back_stacked, which read the ranks'
// addresses off one tensor per argument.
//
// What the reference does not have: World (the expert-parallel world as logical ranks
// of one GPU; Buffer takes the one it belongs to as an optional fifth argument and
// otherwise joins a process-wide world of its num_ranks) and the whole-world calls.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/ones.h>
#include <c10/core/Storage.h>
#include <c10/core/TensorImpl.h>
#include <pybind11/functional.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include <atomic>
#include <climits>
#include <cstdint>
#include <deque>
#include <functional>
#include <map>
#include <memory>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "mooncake_ep_hip.h"

namespace py = pybind11;

namespace {

// EPException surfaces as RuntimeError through pybind11 in the reference; the paths
// its Python wrapper answers with NotImplementedError do so here too.
void check(int rc) {
    if (rc == MC_EP_OK) return;
    const char* msg = mc_ep_last_error();
    if (rc == MC_EP_ERR_UNSUPPORTED) {
        PyErr_SetString(PyExc_NotImplementedError, msg ? msg : "unsupported");
        throw py::error_already_set();
    }
    if (rc == MC_EP_ERR_INVALID) throw std::invalid_argument(msg ? msg : "invalid argument");   // ValueError
    if (rc == MC_EP_ERR_PENDING) {
        // a RuntimeError of its own, shared with the ctypes binding: callers tell "not every rank has called
        // yet" (the call stays posted) from a failure by the type, not by the text
        const std::string text = msg ? msg : "pending";
        py::object type = py::module_::import("mooncake_amd._lib").attr("PendingError");
        PyErr_SetString(type.ptr(), text.c_str());
        throw py::error_already_set();
    }
    throw std::runtime_error(msg ? msg : "mooncake_ep_hip: unknown failure");
}

using U64s = std::vector<uint64_t>;
using I32s = std::vector<int32_t>;

struct World {
    mc_ep_world_t* h = nullptr;
    int num_ranks = 0;
    explicit World(int n) : num_ranks(n) { check(mc_ep_world_create(n, &h)); }
    World(const World&) = delete;
    World& operator=(const World&) = delete;
    ~World() {
        if (h) mc_ep_world_destroy(h);
    }
    void need(const U64s& v, const char* what) const {
        if ((int)v.size() != num_ranks)
            throw std::invalid_argument(std::string(what) + ": one entry per logical rank expected");
    }
};

using WorldPtr = std::shared_ptr<World>;

// Buffers created without a world share one per num_ranks, like processes that join one group.
std::map<int, std::weak_ptr<World>>& default_worlds() {
    static std::map<int, std::weak_ptr<World>> worlds;
    return worlds;
}

WorldPtr default_world(int num_ranks) {
    auto& slot = default_worlds()[num_ranks];
    WorldPtr w = slot.lock();
    if (!w) {
        w = std::make_shared<World>(num_ranks);
        slot = w;
    }
    return w;
}

// EventHandle, mooncake_ep_event.h:9-42
struct Event {
    mc_ep_event_t* h = nullptr;
    WorldPtr keep;   // an event of a collective refers to its world's bookkeeping
    explicit Event(uint64_t stream_ptr) { check(mc_ep_event_create(stream_ptr, &h)); }
    Event(mc_ep_event_t* raw, WorldPtr w) : h(raw), keep(std::move(w)) {}
    Event(const Event&) = delete;
    Event& operator=(const Event&) = delete;
    ~Event() { mc_ep_event_destroy(h); }
    void current_stream_wait(uint64_t stream_ptr) { check(mc_ep_event_current_stream_wait(h, stream_ptr)); }
    void synchronize() { check(mc_ep_event_synchronize(h)); }
};

using CallResult = std::tuple<std::optional<std::shared_ptr<Event>>, std::optional<std::function<void()>>>;

CallResult wrap(mc_ep_event_t* ev, mc_ep_hook_t* hook, const WorldPtr& world) {
    CallResult r;
    if (ev) std::get<0>(r) = std::make_shared<Event>(ev, world);
    if (hook) {
        std::shared_ptr<mc_ep_hook_t> keep(hook, mc_ep_hook_destroy);
        WorldPtr w = world;   // the hook enqueues work of its world: keep it alive
        std::get<1>(r) = [keep, w] { check(mc_ep_hook_call(keep.get())); };
    }
    return r;
}

// A per-rank call may wait for other Python threads (one per rank, option "blocking" - which can be set
// through any binding of the C ABI, so nothing here tries to know): it always gives up the GIL for its
// duration.  The library reports its failure per thread, so the error text is still this call's.
template <typename F>
int without_gil(F&& f) {
    py::gil_scoped_release release;
    return f();
}

// the reference wrapper's checks are Python assertions (mooncake_ep_buffer.py:378-393, :554-567, :616-640)
#define MC_CHECK(cond)                                 \
    do {                                               \
        if (!(cond)) {                                 \
            PyErr_SetString(PyExc_AssertionError, #cond); \
            throw py::error_already_set();             \
        }                                              \
    } while (0)

const at::Tensor& tensor_of(const py::handle& h) {
    if (!THPVariable_Check(h.ptr())) throw py::type_error("a torch.Tensor expected");
    return THPVariable_Unpack(h.ptr());
}

py::object wrap_tensor(at::Tensor t) {
    PyObject* o = THPVariable_Wrap(std::move(t));
    if (o == nullptr) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(o);
}

// torch.empty, with its own exception where memory runs out
at::Tensor empty(c10::IntArrayRef sizes, at::ScalarType type, const at::Device& device) {
    try {
        return at::empty(sizes, at::TensorOptions().dtype(type).device(device));
    } catch (const c10::OutOfMemoryError& e) {
        py::object type = py::module_::import("torch").attr("OutOfMemoryError");
        PyErr_SetString(type.ptr(), e.what_without_backtrace());
        throw py::error_already_set();
    }
}

// sizes travel as int from here on; a larger one is refused as pybind11 refuses it
int as_int(int64_t v) {
    if (v < INT_MIN || v > INT_MAX) throw py::type_error("size out of range");
    return (int)v;
}

uint64_t address(const at::Tensor& t) { return (uint64_t)(uintptr_t)t.data_ptr(); }

// The outputs of earlier dispatches, offered again under the rule of the Python `_OutputPool`: a set is free when
// nothing but the pool refers to any of its storages (tensors, views and dtype reinterpretations of one all do).
// Kept are the storages, not the tensors: every call gets tensors of its own.  Sets are kept per shape, type, device
// and current stream, at most kSets of them per key; a caller that keeps every output alive pools nothing.
class OutputPool {
   public:
    struct Spec {
        std::vector<int64_t> sizes;
        at::ScalarType type;
        std::vector<int64_t> strides = {};   // empty: contiguous
    };
    using Key = std::tuple<int64_t, int64_t, int64_t, bool, int, uint64_t>;

    std::vector<at::Tensor> take(const Key& key, const std::vector<Spec>& specs, const at::Device& device) {
        std::vector<Set>& sets = sets_[key];
        const auto idle = [&](const Set& set) {
            for (size_t i = 0; i < specs.size(); ++i)
                if (set[i].use_count() != 1 || set[i].nbytes() != bytes(specs[i])) return false;
            return true;
        };
        Set fresh;
        const Set* set = nullptr;
        for (size_t i = 0; i < sets.size() && set == nullptr; ++i)
            if (idle(sets[i])) set = &sets[i];
        if (set == nullptr) {
            // outputs are not cleared: rows at and beyond packed_recv_count stay unwritten
            for (const Spec& s : specs) fresh.push_back(empty(s.sizes, s.type, device).storage());
            if (sets.size() < kSets) sets.push_back(fresh);
            set = &fresh;
        }
        std::vector<at::Tensor> out;
        out.reserve(specs.size());
        for (size_t i = 0; i < specs.size(); ++i) {
            const auto dispatch_key = c10::computeDispatchKey(specs[i].type, c10::nullopt, device);
            at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(
                c10::Storage((*set)[i]), c10::DispatchKeySet(dispatch_key), c10::scalarTypeToTypeMeta(specs[i].type));
            if (specs[i].strides.empty()) t.unsafeGetTensorImpl()->set_sizes_contiguous(specs[i].sizes);
            else t.unsafeGetTensorImpl()->set_sizes_and_strides(specs[i].sizes, specs[i].strides);
            out.push_back(std::move(t));
        }
        return out;
    }

   private:
    static constexpr size_t kSets = 4;
    using Set = std::vector<c10::Storage>;
    std::map<Key, std::vector<Set>> sets_;
    static size_t bytes(const Spec& s) {
        size_t n = c10::elementSize(s.type);
        for (int64_t d : s.sizes) n *= (size_t)d;
        return n;
    }
};

// MooncakeEpBuffer, mooncake_ep_buffer.h:66-194
struct Buffer {
    OutputPool outputs;
    mc_ep_buffer_t* h = nullptr;
    WorldPtr world;
    int rank = 0, num_ranks = 0;
    Buffer(int rank_, int num_ranks_, int64_t num_ep_buffer_bytes, bool disable_p2p, WorldPtr w)
        : world(w ? std::move(w) : default_world(num_ranks_)), rank(rank_), num_ranks(num_ranks_) {
        if (world->num_ranks != num_ranks)
            throw std::runtime_error("world has " + std::to_string(world->num_ranks) + " ranks, Buffer asked for " +
                                     std::to_string(num_ranks));
        check(mc_ep_buffer_create(world->h, rank, num_ep_buffer_bytes, disable_p2p ? 1 : 0, &h));
    }
    Buffer(const Buffer&) = delete;
    Buffer& operator=(const Buffer&) = delete;
    ~Buffer() { mc_ep_buffer_destroy(h); }

    // A round's kernels are enqueued by the call of its last rank, from the raw addresses every rank
    // posted, so a call's tensors must outlive the call: whatever the caller hands over as `keep_alive`
    // (the reference's tensors_to_record) is held here until the library reports that the call's round
    // has been enqueued - also when the call itself gave up waiting for its peers (MC_EP_ERR_PENDING:
    // it stays posted).  kind 0: dispatch, 1: combine.  The GIL is held.
    std::deque<py::object> kept[2];
    void retain(int kind, int rc, py::object& keep_alive) {
        if (keep_alive.is_none() || (rc != MC_EP_OK && rc != MC_EP_ERR_PENDING)) return;
        kept[kind].push_back(std::move(keep_alive));
        int pending[2] = {0, 0};
        if (mc_ep_buffer_pending_calls(h, &pending[0], &pending[1]) != MC_EP_OK) return;
        while ((long long)kept[kind].size() > pending[kind]) kept[kind].pop_front();
    }
    std::pair<int, int> retained() const { return {(int)kept[0].size(), (int)kept[1].size()}; }

    CallResult dispatch(uint64_t x_ptr, uint64_t topk_idx_ptr, uint64_t active_ranks_ptr, int num_tokens, int hidden,
                        int num_topk, int num_max_dispatch_tokens_per_rank, int num_experts, int timeout_us,
                        bool use_fp8, uint64_t packed_recv_x_ptr, uint64_t packed_recv_x_scales_ptr,
                        uint64_t packed_recv_count_ptr, uint64_t packed_recv_src_info_ptr,
                        uint64_t packed_recv_layout_range_ptr, bool async, bool return_recv_hook,
                        uint64_t compute_stream_ptr, py::object keep_alive) {
        mc_ep_event_t* ev = nullptr;
        mc_ep_hook_t* hook = nullptr;
        const auto call = [&] {
            return mc_ep_buffer_dispatch(h, x_ptr, topk_idx_ptr, active_ranks_ptr, num_tokens, hidden, num_topk,
                                         num_max_dispatch_tokens_per_rank, num_experts, timeout_us, use_fp8 ? 1 : 0,
                                         packed_recv_x_ptr, packed_recv_x_scales_ptr, packed_recv_count_ptr,
                                         packed_recv_src_info_ptr, packed_recv_layout_range_ptr, async ? 1 : 0,
                                         return_recv_hook ? 1 : 0, compute_stream_ptr, &ev, &hook);
        };
        const int rc = without_gil(call);
        retain(0, rc, keep_alive);
        check(rc);
        return wrap(ev, hook, world);
    }

    CallResult combine(uint64_t x_ptr, uint64_t topk_idx_ptr, uint64_t topk_weights_ptr, uint64_t src_info_ptr,
                       uint64_t layout_range_ptr, uint64_t active_ranks_ptr, int num_local_experts,
                       int num_combined_tokens, int hidden, int num_topk, int num_max_dispatch_tokens_per_rank,
                       int num_experts, int timeout_us, bool zero_copy, uint64_t combined_x_ptr, bool async,
                       bool return_recv_hook, uint64_t compute_stream_ptr, py::object keep_alive) {
        mc_ep_event_t* ev = nullptr;
        mc_ep_hook_t* hook = nullptr;
        const auto call = [&] {
            return mc_ep_buffer_combine(h, x_ptr, topk_idx_ptr, topk_weights_ptr, src_info_ptr, layout_range_ptr,
                                        active_ranks_ptr, num_local_experts, num_combined_tokens, hidden, num_topk,
                                        num_max_dispatch_tokens_per_rank, num_experts, timeout_us, zero_copy ? 1 : 0,
                                        combined_x_ptr, async ? 1 : 0, return_recv_hook ? 1 : 0, compute_stream_ptr,
                                        &ev, &hook);
        };
        const int rc = without_gil(call);
        retain(1, rc, keep_alive);
        check(rc);
        return wrap(ev, hook, world);
    }

    // the rank's view of live ranks: the caller's, or (none given, or one of another size) all of them
    at::Tensor active_or_default(const py::object& active_ranks, const at::Tensor& like) const {
        if (!active_ranks.is_none()) {
            const at::Tensor& active = tensor_of(active_ranks);
            MC_CHECK(active.dim() == 1 && active.is_contiguous());
            MC_CHECK(active.scalar_type() == at::kInt);
            if (active.numel() == num_ranks) return active;
        }
        return at::ones({num_ranks}, at::TensorOptions().dtype(at::kInt).device(like.device()));
    }

    // -> (event, hook, (x, topk_idx, active_ranks, packed_recv_x, scales or None, count, src_info, layout_range))
    py::tuple dispatch_tensors(py::object x_, py::object topk_idx_, py::object active_ranks_, int max_tokens,
                               int num_experts, int timeout_us, bool use_fp8, bool async, bool return_recv_hook,
                               uint64_t stream_ptr) {
        const at::Tensor &x = tensor_of(x_), &topk_idx = tensor_of(topk_idx_);
        MC_CHECK(x.dim() == 2 && x.is_contiguous());
        MC_CHECK(x.scalar_type() == at::kBFloat16);
        MC_CHECK(topk_idx.dim() == 2 && topk_idx.is_contiguous());
        MC_CHECK(topk_idx.scalar_type() == at::kLong);
        const int64_t num_tokens = x.size(0), hidden = x.size(1);
        MC_CHECK(num_tokens == topk_idx.size(0));
        MC_CHECK(num_tokens <= max_tokens);
        MC_CHECK(hidden % 16 == 0 && hidden % 128 == 0);
        MC_CHECK(num_experts % num_ranks == 0);
        const at::Tensor active = active_or_default(active_ranks_, x);
        const int64_t local = num_experts / num_ranks, rm = (int64_t)num_ranks * max_tokens;
        if (use_fp8) MC_CHECK(rm % 4 == 0);

        std::vector<OutputPool::Spec> specs{{{local, rm, hidden}, use_fp8 ? at::kFloat8_e4m3fn : at::kBFloat16},
                                            {{local}, at::kInt},
                                            {{local, rm}, at::kInt},
                                            {{local, (int64_t)num_ranks}, at::kLong}};
        // column-major per expert: [L, H/128, R*max] storage viewed as [L, R*max, H/128]
        if (use_fp8) specs.push_back({{local, rm, hidden / 128}, at::kFloat, {hidden / 128 * rm, 1, rm}});
        std::vector<at::Tensor> outs =
            outputs.take({local, rm, hidden, use_fp8, x.device().index(), stream_ptr}, specs, x.device());
        const uint64_t recv_x = address(outs[0]), count = address(outs[1]), info = address(outs[2]),
                       range = address(outs[3]), scales = use_fp8 ? address(outs[4]) : 0;
        py::object active_obj = active_ranks_;
        if (active_ranks_.is_none() || !active.is_same(tensor_of(active_ranks_))) active_obj = wrap_tensor(active);
        const int num_topk = as_int(topk_idx.size(1));
        const uint64_t x_ptr = address(x), idx_ptr = address(topk_idx), active_ptr = address(active);
        py::tuple kept = py::make_tuple(
            std::move(x_), std::move(topk_idx_), std::move(active_obj), wrap_tensor(std::move(outs[0])),
            use_fp8 ? wrap_tensor(std::move(outs[4])) : py::object(py::none()), wrap_tensor(std::move(outs[1])),
            wrap_tensor(std::move(outs[2])), wrap_tensor(std::move(outs[3])));
        CallResult r = dispatch(x_ptr, idx_ptr, active_ptr, as_int(num_tokens), as_int(hidden), num_topk, max_tokens,
                                num_experts, timeout_us, use_fp8, recv_x, scales, count, info, range, async,
                                return_recv_hook, stream_ptr, kept);
        return py::make_tuple(std::move(std::get<0>(r)), std::move(std::get<1>(r)), std::move(kept));
    }

    // -> (event, hook, (x, topk_idx, topk_weights, active_ranks, src_info, layout_range, combined_x))
    py::tuple combine_tensors(py::object x_, py::object topk_idx_, py::object topk_weights_, py::object active_ranks_,
                              py::object src_info_, py::object layout_range_, int max_tokens, int hidden,
                              int num_experts, int timeout_us, py::object out_, bool async, bool return_recv_hook,
                              uint64_t stream_ptr) {
        const at::Tensor &x = tensor_of(x_), &topk_idx = tensor_of(topk_idx_), &topk_weights = tensor_of(topk_weights_);
        const at::Tensor &src_info = tensor_of(src_info_), &layout_range = tensor_of(layout_range_);
        MC_CHECK(x.dim() == 3 && x.is_contiguous());
        MC_CHECK(x.scalar_type() == at::kBFloat16);
        MC_CHECK(topk_idx.dim() == 2 && topk_idx.is_contiguous());
        MC_CHECK(topk_idx.scalar_type() == at::kLong);
        MC_CHECK(topk_weights.dim() == 2 && topk_weights.is_contiguous());
        MC_CHECK(topk_weights.scalar_type() == at::kFloat);
        const at::Tensor active = active_or_default(active_ranks_, x);
        const int64_t local = num_experts / num_ranks;
        MC_CHECK(x.size(0) == local);
        MC_CHECK(x.size(1) == (int64_t)num_ranks * max_tokens);
        MC_CHECK(x.size(2) == hidden);
        MC_CHECK(hidden % 16 == 0 && hidden % 128 == 0);
        MC_CHECK(topk_idx.sizes() == topk_weights.sizes());
        const int64_t num_tokens = topk_weights.size(0);
        MC_CHECK(num_tokens <= max_tokens);
        MC_CHECK(src_info.dim() == 2 && src_info.is_contiguous());
        MC_CHECK(src_info.scalar_type() == at::kInt);
        MC_CHECK(src_info.size(0) == x.size(0));
        MC_CHECK(layout_range.dim() == 2 && layout_range.is_contiguous());
        MC_CHECK(layout_range.scalar_type() == at::kLong);
        MC_CHECK(layout_range.size(0) == local);
        MC_CHECK(layout_range.size(1) == num_ranks);
        at::Tensor combined;
        if (!out_.is_none()) {
            combined = tensor_of(out_);
            MC_CHECK(combined.dim() == 2 && combined.is_contiguous());
            MC_CHECK(combined.size(0) == num_tokens);
            MC_CHECK(combined.size(1) == hidden);
            MC_CHECK(combined.scalar_type() == at::kBFloat16);
        } else {
            combined = empty({num_tokens, hidden}, at::kBFloat16, x.device());
            out_ = wrap_tensor(combined);
        }
        py::object active_obj = active_ranks_;
        if (active_ranks_.is_none() || !active.is_same(tensor_of(active_ranks_))) active_obj = wrap_tensor(active);
        const uint64_t x_ptr = address(x), idx_ptr = address(topk_idx), weights_ptr = address(topk_weights),
                       info_ptr = address(src_info), range_ptr = address(layout_range), active_ptr = address(active),
                       out_ptr = address(combined);
        const int num_topk = as_int(topk_weights.size(1));
        py::tuple kept = py::make_tuple(std::move(x_), std::move(topk_idx_), std::move(topk_weights_),
                                        std::move(active_obj), std::move(src_info_), std::move(layout_range_),
                                        std::move(out_));
        CallResult r = combine(x_ptr, idx_ptr, weights_ptr, info_ptr, range_ptr, active_ptr, as_int(local), as_int(num_tokens),
                               hidden, num_topk, max_tokens, num_experts, timeout_us, false, out_ptr, async,
                               return_recv_hook, stream_ptr, kept);
        return py::make_tuple(std::move(std::get<0>(r)), std::move(std::get<1>(r)), std::move(kept));
    }

    std::pair<int, int> pending_calls() const {
        int d = 0, c = 0;
        check(mc_ep_buffer_pending_calls(h, &d, &c));
        return {d, c};
    }
};

// A whole-world call whose per-rank address arrays were marshalled once.
struct PreparedDispatch {
    WorldPtr world;
    U64s x, topk_idx, recv_x, recv_scales, recv_count, src_info, layout_range;
    I32s num_tokens;
    int hidden = 0, num_topk = 0, max_tokens = 0, num_experts = 0, use_fp8 = 0;
    void call(uint64_t stream_ptr, int phases) const {
        check(mc_ep_world_dispatch(world->h, x.data(), topk_idx.data(), num_tokens.data(), hidden, num_topk, max_tokens,
                                   num_experts, use_fp8, recv_x.data(), use_fp8 ? recv_scales.data() : nullptr,
                                   recv_count.data(), src_info.data(), layout_range.data(), phases, stream_ptr));
    }
    void call_noalloc(uint64_t stream_ptr) const {
        check(mc_ep_world_dispatch_noalloc(world->h, x.data(), topk_idx.data(), num_tokens.data(), hidden, num_topk,
                                           max_tokens, num_experts, use_fp8, recv_x.data(),
                                           use_fp8 ? recv_scales.data() : nullptr, recv_count.data(), src_info.data(),
                                           layout_range.data(), stream_ptr));
    }
};

struct PreparedCombine {
    WorldPtr world;
    U64s x, scales, topk_idx, topk_weights, src_info, layout_range, active_ranks, out;
    I32s num_tokens;
    uint64_t factor = 0;
    bool packed = false, has_scales = false;
    int hidden = 0, num_topk = 0, max_tokens = 0, num_experts = 0;
    void call(uint64_t stream_ptr, int phases) const {
        if (packed)
            check(mc_ep_world_combine_packed(world->h, x.data(), has_scales ? scales.data() : nullptr, factor,
                                             topk_idx.data(), topk_weights.data(), src_info.data(),
                                             layout_range.data(), active_ranks.data(), num_tokens.data(), hidden,
                                             num_topk, max_tokens, num_experts, out.data(), phases, stream_ptr));
        else
            check(mc_ep_world_combine(world->h, x.data(), topk_idx.data(), topk_weights.data(), src_info.data(),
                                      layout_range.data(), active_ranks.data(), num_tokens.data(), hidden, num_topk,
                                      max_tokens, num_experts, out.data(), phases, stream_ptr));
    }
};

// The whole-world calls from stacked tensors: rank r's tensor is slice r of one tensor, and its address, which indexing in
// Python costs 0.4 us to learn, is the first one's plus r strides.  Everything is read off the tensors at each call and
// nothing kept.  A call answers false, having done nothing, where a tensor is neither None nor a plain torch.Tensor (or
// Parameter; another subclass may have its own idea of indexing) with a slice per rank, or the token counts or
// the ranks that take part are not plain lists: the caller then marshals it in Python, or is refused there.
// Host time of a call, us (of two speeds that one host ran at): 4 ranks, dispatch and combine 5.2 to 6.1 -> 4.0 to 4.9
// (keyed and looked up in Python before), cast back 16 to 17 -> 4.5 to 5.8 (a slice per rank and tensor before); 32 ranks,
// dispatch 10.7 to 12.9 -> 7.3 to 9.9, combine 5.8 to 7.2 -> 4.7 to 6.5, cast back 120 -> 4.8 to 6.6.
class Stacked {
   public:
    explicit Stacked(const World& w) : ranks_(w.num_ranks) { words_.reserve((size_t)8 * ranks_); }

    // Every step below answers false where it is given anything but the plain form.  No Python code runs in between (a
    // list's items are looked at only where they are plain numbers), so nothing can change under it.

    // which ranks take part (None: all): a list or a tuple of numbers, one per rank
    bool take_part(const py::handle& present) {
        if (present.is_none()) return true;
        PyObject* p = present.ptr();
        const bool list = PyList_CheckExact(p);
        if (!(list || PyTuple_CheckExact(p)) || Py_SIZE(p) != ranks_) return false;
        present_.resize(ranks_);
        for (int r = 0; r < ranks_; ++r) {
            PyObject* on = list ? PyList_GET_ITEM(p, r) : PyTuple_GET_ITEM(p, r);
            if (!PyBool_Check(on) && !PyLong_CheckExact(on)) return false;
            present_[r] = PyObject_IsTrue(on) != 0;
        }
        return true;
    }
    // and, of those, how many tokens: a list of numbers, one per rank
    bool tokens(const py::handle& counts) {
        if (!PyList_CheckExact(counts.ptr()) || PyList_GET_SIZE(counts.ptr()) != ranks_) return false;
        counts_.resize(ranks_);
        for (int r = 0; r < ranks_; ++r) {
            PyObject* n = PyList_GET_ITEM(counts.ptr(), r);
            int overflow = 0;
            const long v = PyLong_CheckExact(n) ? PyLong_AsLongAndOverflow(n, &overflow) : -1;
            if (overflow != 0 || v < 0 || v > INT_MAX) return false;
            counts_[r] = (!present_.empty() && !present_[r]) ? 0 : (int)v;
        }
        return true;
    }
    // a tensor's addresses (zeros for None, and, of_present, for ranks that take no part)
    bool add(const py::handle& h, bool of_present = false) {
        const size_t at = words_.size();
        words_.resize(at + ranks_, 0);
        if (h.is_none()) return true;
        if (!THPVariable_CheckExact(h.ptr())) return false;
        const at::Tensor& t = THPVariable_Unpack(h.ptr());
        if (t.layout() != at::kStrided || t.dim() < 1 || t.size(0) < ranks_) return false;
        if (t.numel() == 0) return true;               // (an empty tensor has no address)
        const uint64_t first = address(t);
        const int64_t step = t.stride(0) * (int64_t)t.element_size();
        for (int r = 0; r < ranks_; ++r)
            if (!of_present || present_.empty() || present_[r]) words_[at + r] = first + (uint64_t)(step * r);
        return true;
    }
    const uint64_t* operator[](int i) const { return words_.data() + (size_t)i * ranks_; }
    const int32_t* counts() const { return counts_.data(); }

   private:
    int ranks_;
    U64s words_;
    I32s counts_;
    std::vector<char> present_;
};

bool dispatch_stacked(const World& w, py::handle x, py::handle topk_idx, py::handle recv_x, py::handle recv_scales,
                      py::handle recv_count, py::handle src_info, py::handle layout_range, py::handle num_tokens,
                      py::handle present, int hidden, int num_topk, int max_tokens, int num_experts, bool use_fp8,
                      int phases, uint64_t stream_ptr) {
    Stacked s(w);
    if (!s.take_part(present) || !s.tokens(num_tokens) || !s.add(x) || !s.add(topk_idx) || !s.add(recv_x, true) ||
        !s.add(recv_scales, true) || !s.add(recv_count, true) || !s.add(src_info, true) || !s.add(layout_range, true))
        return false;
    check(mc_ep_world_dispatch(w.h, s[0], s[1], s.counts(), hidden, num_topk, max_tokens, num_experts, use_fp8 ? 1 : 0,
                               s[2], use_fp8 ? s[3] : nullptr, s[4], s[5], s[6], phases, stream_ptr));
    return true;
}

// packed: x is the payload dispatch wrote (scales None: bf16), factor_ptr a factor per expert (0: none)
bool combine_stacked(const World& w, py::handle x, py::handle scales, py::handle topk_idx, py::handle topk_weights,
                     py::handle src_info, py::handle layout_range, py::handle active_ranks, py::handle out,
                     py::handle num_tokens, py::handle present, int hidden, int num_topk, int max_tokens, int num_experts,
                     bool packed, uint64_t factor_ptr, int phases, uint64_t stream_ptr) {
    Stacked s(w);
    if (!s.take_part(present) || !s.tokens(num_tokens) || !s.add(x, true) || !s.add(scales, true) || !s.add(topk_idx) ||
        !s.add(topk_weights) || !s.add(src_info) || !s.add(layout_range) || !s.add(active_ranks) || !s.add(out))
        return false;
    if (packed)
        check(mc_ep_world_combine_packed(w.h, s[0], scales.is_none() ? nullptr : s[1], factor_ptr, s[2], s[3], s[4], s[5],
                                         s[6], s.counts(), hidden, num_topk, max_tokens, num_experts, s[7], phases,
                                         stream_ptr));
    else
        check(mc_ep_world_combine(w.h, s[0], s[2], s[3], s[4], s[5], s[6], s.counts(), hidden, num_topk, max_tokens,
                                  num_experts, s[7], phases, stream_ptr));
    return true;
}

bool cast_back_stacked(const World& w, py::handle recv_x, py::handle scales, py::handle recv_count, uint64_t factor_ptr,
                       py::handle out, py::handle present, int hidden, int num_topk, int max_tokens, int num_experts,
                       uint64_t stream_ptr) {
    Stacked s(w);
    if (!s.take_part(present) || !s.add(recv_x, true) || !s.add(scales, true) || !s.add(recv_count) || !s.add(out))
        return false;
    check(mc_ep_world_cast_back(w.h, s[0], scales.is_none() ? nullptr : s[1], s[2], factor_ptr, s[3], hidden, num_topk,
                                max_tokens, num_experts, stream_ptr));
    return true;
}

// LegacyBufferPerfTensors / Config / Result of legacy_buffer_perf.cpp:18-49, with one device address
// per logical rank where the reference has one address.
struct LegacyTensors {
    U64s x_ptr, topk_idx_ptr, topk_weights_ptr, active_ranks_ptr, expert_x_ptr, packed_recv_x_ptr,
        packed_recv_count_ptr, packed_recv_src_info_ptr, packed_recv_layout_range_ptr, combined_x_ptr;
};

struct LegacyConfig {
    int num_tokens = 0, hidden = 0, num_topk = 0, num_local_experts = 0, num_max_dispatch_tokens_per_rank = 0,
        num_experts = 0, timeout_us = -1, warmups = 20, iterations = 30;
    uint64_t compute_stream_ptr = 0;
};

struct LegacyResult {
    double average_us = 0.0, min_us = 0.0, max_us = 0.0;
};

LegacyResult benchmark_legacy(const WorldPtr& world, const LegacyTensors& t, const LegacyConfig& c) {
    const U64s* fields[] = {&t.x_ptr,           &t.topk_idx_ptr,          &t.topk_weights_ptr,
                            &t.active_ranks_ptr, &t.expert_x_ptr,          &t.packed_recv_x_ptr,
                            &t.packed_recv_count_ptr, &t.packed_recv_src_info_ptr,
                            &t.packed_recv_layout_range_ptr, &t.combined_x_ptr};
    for (const U64s* f : fields)
        if ((int)f->size() != world->num_ranks)
            throw std::invalid_argument("legacy EP benchmark received a null tensor pointer");
    mc_ep_legacy_perf_tensors_t ct{t.x_ptr.data(),
                                   t.topk_idx_ptr.data(),
                                   t.topk_weights_ptr.data(),
                                   t.active_ranks_ptr.data(),
                                   t.expert_x_ptr.data(),
                                   t.packed_recv_x_ptr.data(),
                                   t.packed_recv_count_ptr.data(),
                                   t.packed_recv_src_info_ptr.data(),
                                   t.packed_recv_layout_range_ptr.data(),
                                   t.combined_x_ptr.data()};
    mc_ep_legacy_perf_config_t cc{c.num_tokens, c.hidden,     c.num_topk,   c.num_local_experts,
                                  c.num_max_dispatch_tokens_per_rank, c.num_experts, c.timeout_us,
                                  c.warmups,    c.iterations, c.compute_stream_ptr};
    mc_ep_legacy_perf_result_t cr{0, 0, 0};
    int rc;
    {
        py::gil_scoped_release release;   // as the reference's binding does for its timed loop
        rc = mc_ep_world_legacy_buffer_perf(world->h, &ct, &cc, &cr);
    }
    check(rc);
    return LegacyResult{cr.average_us, cr.min_us, cr.max_us};
}

}  // namespace

PYBIND11_MODULE(_ep, m) {
    m.doc() = "Low-latency MoE dispatch / combine on one AMD MI355X (C ABI: include/mooncake_ep_hip.h)";
    m.def("get_ep_buffer_size_hint", [](int max_tokens, int hidden, int num_ranks, int num_experts) {
        return mc_ep_get_buffer_size_hint(max_tokens, hidden, num_ranks, num_experts);
    });
    m.attr("MAX_QP_COUNT") = py::int_(MC_EP_MAX_QP_COUNT);
    m.attr("PHASE_LAYOUT") = py::int_(MC_EP_PHASE_LAYOUT);
    m.attr("PHASE_DATA") = py::int_(MC_EP_PHASE_DATA);
    m.attr("PHASE_FINISH") = py::int_(MC_EP_PHASE_FINISH);
    m.attr("PHASE_ALL") = py::int_(MC_EP_PHASE_ALL);

    py::class_<Event, std::shared_ptr<Event>>(m, "EventHandle")
        .def(py::init<uint64_t>(), py::arg("stream_ptr") = 0)
        .def("current_stream_wait", &Event::current_stream_wait, py::arg("stream_ptr"))
        .def("synchronize", &Event::synchronize);

    py::class_<PreparedDispatch>(m, "_PreparedDispatch")
        .def("__call__", &PreparedDispatch::call, py::arg("stream_ptr"), py::arg("phases") = MC_EP_PHASE_ALL)
        .def("noalloc", &PreparedDispatch::call_noalloc, py::arg("stream_ptr"));
    py::class_<PreparedCombine>(m, "_PreparedCombine")
        .def("__call__", &PreparedCombine::call, py::arg("stream_ptr"), py::arg("phases") = MC_EP_PHASE_ALL);

    py::class_<World, WorldPtr>(m, "World")
        .def(py::init<int>(), py::arg("num_ranks"))
        .def_readonly("num_ranks", &World::num_ranks)
        .def_property_readonly("handle", [](const World& w) { return (uintptr_t)w.h; },
                               "address of the mc_ep_world_t, for callers of the C ABI")
        .def("set_rank_silent",
             [](World& w, int rank, bool silent) { check(mc_ep_world_set_rank_silent(w.h, rank, silent ? 1 : 0)); },
             py::arg("rank"), py::arg("silent") = true)
        .def("set_option",
             [](World& w, const std::string& name, int value) {
                 check(mc_ep_world_set_option(w.h, name.c_str(), value));
             })
        .def("get_option",
             [](const World& w, const std::string& name) {
                 int v = 0;
                 check(mc_ep_world_get_option(w.h, name.c_str(), &v));
                 return v;
             })
        .def("prepare_dispatch",
             [](const WorldPtr& w, U64s x, U64s topk_idx, I32s num_tokens, int hidden, int num_topk, int max_tokens,
                int num_experts, bool use_fp8, U64s recv_x, std::optional<U64s> recv_scales, U64s recv_count,
                U64s src_info, U64s layout_range) {
                 PreparedDispatch p;
                 p.world = w;
                 w->need(x, "x_ptrs");
                 w->need(topk_idx, "topk_idx_ptrs");
                 w->need(recv_x, "packed_recv_x_ptrs");
                 w->need(recv_count, "packed_recv_count_ptrs");
                 w->need(src_info, "packed_recv_src_info_ptrs");
                 w->need(layout_range, "packed_recv_layout_range_ptrs");
                 if ((int)num_tokens.size() != w->num_ranks) throw std::invalid_argument("num_tokens: one per rank");
                 if (use_fp8) {
                     if (!recv_scales) throw std::invalid_argument("fp8 dispatch needs packed_recv_x_scales_ptrs");
                     w->need(*recv_scales, "packed_recv_x_scales_ptrs");
                     p.recv_scales = std::move(*recv_scales);
                 }
                 p.x = std::move(x); p.topk_idx = std::move(topk_idx); p.num_tokens = std::move(num_tokens);
                 p.recv_x = std::move(recv_x); p.recv_count = std::move(recv_count);
                 p.src_info = std::move(src_info); p.layout_range = std::move(layout_range);
                 p.hidden = hidden; p.num_topk = num_topk; p.max_tokens = max_tokens; p.num_experts = num_experts;
                 p.use_fp8 = use_fp8 ? 1 : 0;
                 return p;
             })
        .def("prepare_combine",
             [](const WorldPtr& w, U64s x, std::optional<U64s> scales, uint64_t expert_factor_ptr, bool packed,
                U64s topk_idx, U64s topk_weights, U64s src_info, U64s layout_range, U64s active_ranks,
                I32s num_tokens, int hidden, int num_topk, int max_tokens, int num_experts, U64s out) {
                 PreparedCombine p;
                 p.world = w;
                 w->need(x, "x_ptrs");
                 w->need(topk_idx, "topk_idx_ptrs");
                 w->need(topk_weights, "topk_weights_ptrs");
                 w->need(src_info, "src_info_ptrs");
                 w->need(layout_range, "layout_range_ptrs");
                 w->need(active_ranks, "active_ranks_ptrs");
                 w->need(out, "combined_x_ptrs");
                 if ((int)num_tokens.size() != w->num_ranks) throw std::invalid_argument("num_tokens: one per rank");
                 if (scales) {
                     w->need(*scales, "packed_recv_x_scales_ptrs");
                     p.scales = std::move(*scales);
                     p.has_scales = true;
                 }
                 p.packed = packed; p.factor = expert_factor_ptr;
                 p.x = std::move(x); p.topk_idx = std::move(topk_idx); p.topk_weights = std::move(topk_weights);
                 p.src_info = std::move(src_info); p.layout_range = std::move(layout_range);
                 p.active_ranks = std::move(active_ranks); p.out = std::move(out); p.num_tokens = std::move(num_tokens);
                 p.hidden = hidden; p.num_topk = num_topk; p.max_tokens = max_tokens; p.num_experts = num_experts;
                 return p;
             })
        .def("dispatch_stacked", &dispatch_stacked)
        .def("combine_stacked", &combine_stacked)
        .def("cast_back_stacked", &cast_back_stacked)
        .def("cast_back",
             [](const WorldPtr& w, U64s recv_x, std::optional<U64s> recv_scales, U64s recv_count,
                uint64_t expert_factor_ptr, U64s out, int hidden, int num_topk, int max_tokens, int num_experts,
                uint64_t stream_ptr) {
                 w->need(recv_x, "packed_recv_x_ptrs");
                 w->need(recv_count, "packed_recv_count_ptrs");
                 w->need(out, "out_ptrs");
                 if (recv_scales) w->need(*recv_scales, "packed_recv_x_scales_ptrs");
                 check(mc_ep_world_cast_back(w->h, recv_x.data(), recv_scales ? recv_scales->data() : nullptr,
                                             recv_count.data(), expert_factor_ptr, out.data(), hidden, num_topk,
                                             max_tokens, num_experts, stream_ptr));
             });

    py::class_<LegacyTensors>(m, "_LegacyBufferPerfTensors")
        .def(py::init<>())
        .def_readwrite("x_ptr", &LegacyTensors::x_ptr)
        .def_readwrite("topk_idx_ptr", &LegacyTensors::topk_idx_ptr)
        .def_readwrite("topk_weights_ptr", &LegacyTensors::topk_weights_ptr)
        .def_readwrite("active_ranks_ptr", &LegacyTensors::active_ranks_ptr)
        .def_readwrite("expert_x_ptr", &LegacyTensors::expert_x_ptr)
        .def_readwrite("packed_recv_x_ptr", &LegacyTensors::packed_recv_x_ptr)
        .def_readwrite("packed_recv_count_ptr", &LegacyTensors::packed_recv_count_ptr)
        .def_readwrite("packed_recv_src_info_ptr", &LegacyTensors::packed_recv_src_info_ptr)
        .def_readwrite("packed_recv_layout_range_ptr", &LegacyTensors::packed_recv_layout_range_ptr)
        .def_readwrite("combined_x_ptr", &LegacyTensors::combined_x_ptr);
    py::class_<LegacyConfig>(m, "_LegacyBufferPerfConfig")
        .def(py::init<>())
        .def_readwrite("num_tokens", &LegacyConfig::num_tokens)
        .def_readwrite("hidden", &LegacyConfig::hidden)
        .def_readwrite("num_topk", &LegacyConfig::num_topk)
        .def_readwrite("num_local_experts", &LegacyConfig::num_local_experts)
        .def_readwrite("num_max_dispatch_tokens_per_rank", &LegacyConfig::num_max_dispatch_tokens_per_rank)
        .def_readwrite("num_experts", &LegacyConfig::num_experts)
        .def_readwrite("timeout_us", &LegacyConfig::timeout_us)
        .def_readwrite("warmups", &LegacyConfig::warmups)
        .def_readwrite("iterations", &LegacyConfig::iterations)
        .def_readwrite("compute_stream_ptr", &LegacyConfig::compute_stream_ptr);
    py::class_<LegacyResult>(m, "_LegacyBufferPerfResult")
        .def_readonly("average_us", &LegacyResult::average_us)
        .def_readonly("min_us", &LegacyResult::min_us)
        .def_readonly("max_us", &LegacyResult::max_us);

    py::class_<Buffer>(m, "Buffer")
        .def(py::init<int, int, int64_t, bool, WorldPtr>(), py::arg("rank"), py::arg("num_ranks"),
             py::arg("num_ep_buffer_bytes"), py::arg("disable_p2p") = false, py::arg("world") = WorldPtr())
        .def_readonly("world", &Buffer::world)
        .def_readonly("rank", &Buffer::rank)
        .def_readonly("num_ranks", &Buffer::num_ranks)
        // transport introspection (ep_py.cpp:31-42): one address space, no NIC, no peer process
        .def("ibgda_disabled", [](const Buffer& b) { return mc_ep_buffer_ibgda_disabled(b.h) != 0; })
        .def("p2p_enabled", [](const Buffer& b) { return mc_ep_buffer_p2p_enabled(b.h) != 0; })
        .def("use_fast_path", [](const Buffer& b) { return mc_ep_buffer_use_fast_path(b.h) != 0; })
        .def("is_roce", [](const Buffer& b) { return mc_ep_buffer_is_roce(b.h) != 0; })
        .def("update_local_qpns", [](Buffer&) {})
        .def("sync_ibgda_peers", [](Buffer&, py::object, py::object, py::object, py::object, py::object, py::object,
                                    py::object) {})
        .def("get_mr_info", [](const Buffer&) { return std::make_pair<uint64_t, uint32_t>(0, 0); })
        .def("get_gid", [](const Buffer&) { return std::make_pair<uint64_t, uint64_t>(0, 0); })
        .def("get_local_qpns", [](const Buffer&) { return std::vector<int32_t>(); })
        .def("get_local_lids", [](const Buffer&) { return std::vector<int32_t>(); })
        .def("get_ipc_handle", [](const Buffer&) { return std::vector<int32_t>(); })
        .def("sync_nvlink_ipc_handles", [](Buffer&, py::object, py::object) {})
        .def("pending_calls", &Buffer::pending_calls)
        .def("retained", &Buffer::retained, "(dispatch, combine) keep_alive objects still held")
        // what the Python `Buffer`'s dispatch and combine are made of (positional arguments)
        .def("dispatch_tensors", &Buffer::dispatch_tensors)
        .def("combine_tensors", &Buffer::combine_tensors)
        // the reference's argument lists (ep_py.cpp:43-44), positional; keep_alive is this module's addition
        .def("dispatch", &Buffer::dispatch, py::arg("x_ptr"), py::arg("topk_idx_ptr"), py::arg("active_ranks_ptr"),
             py::arg("num_tokens"), py::arg("hidden"), py::arg("num_topk"),
             py::arg("num_max_dispatch_tokens_per_rank"), py::arg("num_experts"), py::arg("timeout_us"),
             py::arg("use_fp8"), py::arg("packed_recv_x_ptr"), py::arg("packed_recv_x_scales_ptr"),
             py::arg("packed_recv_count_ptr"), py::arg("packed_recv_src_info_ptr"),
             py::arg("packed_recv_layout_range_ptr"), py::arg("async"), py::arg("return_recv_hook"),
             py::arg("compute_stream_ptr"), py::arg("keep_alive") = py::none())
        .def("combine", &Buffer::combine, py::arg("x_ptr"), py::arg("topk_idx_ptr"), py::arg("topk_weights_ptr"),
             py::arg("src_info_ptr"), py::arg("layout_range_ptr"), py::arg("active_ranks_ptr"),
             py::arg("num_local_experts"), py::arg("num_combined_tokens"), py::arg("hidden"), py::arg("num_topk"),
             py::arg("num_max_dispatch_tokens_per_rank"), py::arg("num_experts"), py::arg("timeout_us"),
             py::arg("zero_copy"), py::arg("combined_x_ptr"), py::arg("async"), py::arg("return_recv_hook"),
             py::arg("compute_stream_ptr"), py::arg("keep_alive") = py::none());

    m.def("_benchmark_legacy_buffer",
          [](const py::object& runtime, const LegacyTensors& t, const LegacyConfig& c) {
              // the reference passes one rank's Buffer; here the loop drives the Buffer's whole world
              if (py::isinstance<Buffer>(runtime)) return benchmark_legacy(runtime.cast<Buffer&>().world, t, c);
              return benchmark_legacy(runtime.cast<WorldPtr>(), t, c);
          },
          py::arg("runtime"), py::arg("tensors"), py::arg("config"));
}

// Python extension module `GNNAdvisor` for PyTorch-ROCm: the twelve functions the
// reference's Python calls (EPPGCN/GCNConv/EPPGCN.cpp:388-403), same positional
// signatures, implemented over the C ABI of libeppgcn_hip.so.  torch supplies the
// tensors and the current HIP stream (and torch::mm for dense products whose shapes
// the library's tall-and-skinny kernels do not cover); everything else happens in
// the HIP library.  Host C++ only: no device code in this file.
//
// Differences from the reference binding, all deliberate:
//   - errors raise (RuntimeError in Python) instead of printf + exit(-1);
//   - work is issued on torch's current stream and is asynchronous unless a host
//     value is returned;
//   - build_part computes on the device and returns int32 tensors (the reference
//     loops on the CPU and returns float32, which corrupts offsets above 2^24);
//   - compact_back_edge's info tensor is float64 so that int(info[0].item()) is
//     exact for any edge count;
//   - split_back_part's part_pointer has num_edges + 1 entries, so the terminator
//     is always in bounds;
//   - get_map_back_part_size never returns less than 1: where the fitted regression drops below 1
//     (large paths) it returns the group size of the rule fitted for the wave64 kernels;
//   - get_ginfo also accepts a CPU tensor, as the reference's host loop does;
//   - the module keeps, per group array it has seen, a column-blocked execution plan for the
//     aggregation kernels (built on first use, about 4 bytes per edge, the most recently used
//     kept: eight, and more while they are small); it affects speed only.
#include <torch/extension.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <cstddef>
#include <cstdint>
#include <iterator>
#include <list>
#include <utility>
#include <vector>

#include "eppgcn_hip.h"

namespace {

using torch::Tensor;

void check(int rc, const char* what)
{
    TORCH_CHECK(rc == 0, what, " failed (", rc, "): ", eppgcn_last_error());
}

#define CHECK_DEVICE(x) TORCH_CHECK((x).is_cuda(), #x " must be a GPU tensor")
#define CHECK_CONTIGUOUS(x) TORCH_CHECK((x).is_contiguous(), #x " must be contiguous")
#define CHECK_INPUT(x) \
    CHECK_DEVICE(x);   \
    CHECK_CONTIGUOUS(x)
#define CHECK_I32(x) \
    CHECK_INPUT(x);  \
    TORCH_CHECK((x).scalar_type() == torch::kInt32, #x " must be int32")
#define CHECK_F32(x) \
    CHECK_INPUT(x);  \
    TORCH_CHECK((x).scalar_type() == torch::kFloat32, #x " must be float32")
#define CHECK_MASK(x) \
    CHECK_INPUT(x);   \
    TORCH_CHECK((x).scalar_type() == torch::kBool || (x).scalar_type() == torch::kUInt8, #x " must be bool")

// Slots and vertices are int32 on the device, and the kernels step through slot ranges in strides of
// up to 1024 past a group's end before clamping: leave that much headroom below 2^31.
#define CHECK_COUNTS(edges, vertices)                                                                      \
    TORCH_CHECK((edges).numel() <= INT32_MAX - 1024, #edges " holds more slots than int32 indexing allows"); \
    TORCH_CHECK((vertices) <= INT32_MAX - 1024, "more vertices than int32 indexing allows")

void* stream_of(const Tensor& t)
{
    return static_cast<void*>(c10::hip::getCurrentHIPStream(t.get_device()).stream());
}

const int32_t* i32(const Tensor& t) { return t.numel() ? t.data_ptr<int32_t>() : nullptr; }
const float* f32(const Tensor& t) { return t.numel() ? t.data_ptr<float>() : nullptr; }

Tensor workspace(size_t bytes, const Tensor& like)
{
    return torch::empty({static_cast<int64_t>((bytes + 7) / 8)}, like.options().dtype(torch::kInt64));
}

// ---------------------------------------------------------------- plan cache
// The column-blocked execution plan depends only on the groups and the column ids, which a
// training run passes unchanged every epoch.  Entries are keyed by storage address, length,
// tensor version and block-size class; an entry holds its key tensors, or (behind the eight used last) is valid only while
// their storages live, so that an address cannot be reused for other data while its entry is valid.
// Staleness rule: an entry is invalidated by writes that bump torch's version counter (ordinary
// in-place tensor operations).  A writer that bypasses the counter - `.data` / detach() in-place
// operations, a raw-pointer kernel of another extension, this library's own C ABI writing into the
// same storage - leaves the cached plan describing the old groups; after such a write call
// clear_plans() before the next layer operation.
size_t held_bytes(const Tensor& t) { return t.defined() ? t.storage().nbytes() : 0; }

// A key tensor of an entry.  As long as its storage lives, by the entry's hand or by somebody else's, and has the memory it
// had, the address the entry was made for cannot hold other data.  A held tensor alone does not say so: its storage can be
// resized, and it can be given another storage (`.data = ...`).
struct Key {
    Tensor held;
    c10::weak_intrusive_ptr<c10::StorageImpl> storage;
    const void* memory;
    explicit Key(const Tensor& t) : held(t), storage(t.storage().getWeakStorageImpl()), memory(t.storage().data()) {}
    bool alive() const
    {
        const auto s = storage.lock();
        return s && s->data() == memory;
    }
    size_t bytes() const { return held_bytes(held); }
};

struct PlanEntry {
    const void* part_ptr;
    const void* col;
    const void* rows;
    int64_t num_parts;
    int64_t num_nodes;          // the plan's layout depends on it
    int64_t version_part, version_col, version_rows;
    int dim_class;
    Key keep_part, keep_col, keep_rows;
    Tensor plan;
    const void* plan_ptr;
    size_t bytes() const { return keep_part.bytes() + keep_col.bytes() + keep_rows.bytes() + held_bytes(plan); }
    bool alive() const { return keep_part.alive() && keep_col.alive() && keep_rows.alive(); }
    void let_go() { keep_part.held.reset(), keep_col.held.reset(), keep_rows.held.reset(); }
};
std::list<PlanEntry> g_plans;
// What the two caches of this file keep: the eight entries used last, whatever their size, and behind them up to 56 more
// whose key tensors live by their owner's hand, while all of a cache together hold at most 256 MB of device memory.  Eight
// alone were less than the layers of a few live models: three models of four layers trained in turn looked every path over
// again in every backward call, two host waits each - 628 us an epoch at 19 717 vertices instead of 369.
constexpr size_t kAlwaysKept = 8, kMostKept = 64, kKeptBytes = size_t(256) << 20;
template <class Cache, class Drop>
void trim(Cache& cache, const Drop& drop)
{
    size_t bytes = 0, place = 0;
    for (auto it = cache.begin(); it != cache.end();) {
        if (place >= kAlwaysKept) it->let_go();
        const size_t here = it->bytes();
        if (it->alive() && (place < kAlwaysKept || (place < kMostKept && bytes + here <= kKeptBytes))) {
            bytes += here;
            ++place;
            ++it;
        } else {
            drop(*it);
            it = cache.erase(it);
        }
    }
}
// An entry that leaves the cache gives its plan's memory back to torch: the library is told first, so that it
// forgets the header it read at that address.
void trim_plans()
{
    trim(g_plans, [](const PlanEntry& e) { eppgcn_plan_release(e.plan_ptr); });
}
void drop_all_plans()
{
    for (const PlanEntry& e : g_plans) eppgcn_plan_release(e.plan_ptr);
    g_plans.clear();
}
int g_plan_policy = 0;   // 0: where eppgcn_plan_recommended says so, 1: always, -1: never

int dim_class_of(int dim) { return dim <= 32 ? 0 : dim <= 128 ? 1 : 2; }
int dim_of_class(int c) { return c == 0 ? 32 : c == 1 ? 128 : 256; }

Tensor aligned_bytes(size_t bytes, const Tensor& like, void** base)
{
    auto t = torch::empty({static_cast<int64_t>(bytes + 256)}, like.options().dtype(torch::kUInt8));
    *base = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(t.data_ptr()) + 255) / 256 * 256);
    return t;
}

// rows: part2Node (forward groups, is_forward) or the per-edge id list (backward path);
// num_slots < 0: read it from part_ptr[num_parts] when the plan has to be built
const void* plan_for(const Tensor& part_ptr, const Tensor& col, const Tensor& rows, bool is_forward, int64_t num_parts,
                     int64_t num_slots, int num_nodes, int dim, int block_shift = 0)
{
    if (num_parts <= 0 || g_plan_policy < 0) return nullptr;
    if (g_plan_policy == 0 && !eppgcn_plan_recommended(num_nodes, dim)) return nullptr;
    const int dc = dim_class_of(dim);
    for (auto it = g_plans.begin(); it != g_plans.end(); ++it) {
        if (it->part_ptr == part_ptr.data_ptr() && it->col == col.data_ptr() && it->rows == rows.data_ptr() &&
            it->num_parts == num_parts && it->num_nodes == num_nodes && it->dim_class == dc &&
            it->version_part == static_cast<int64_t>(part_ptr._version()) &&
            it->version_col == static_cast<int64_t>(col._version()) &&
            it->version_rows == static_cast<int64_t>(rows._version()) && it->alive()) {
            if (it != g_plans.begin()) {                    // most recently used first
                it->keep_part.held = part_ptr, it->keep_col.held = col, it->keep_rows.held = rows;
                g_plans.splice(g_plans.begin(), g_plans, it);
                if (g_plans.size() > kAlwaysKept) std::next(g_plans.begin(), kAlwaysKept)->let_go();
            }
            return g_plans.front().plan_ptr;
        }
    }
    if (num_slots < 0) num_slots = part_ptr[num_parts].item<int64_t>();   // slots the groups cover (one 4-byte read)
    PlanEntry e{part_ptr.data_ptr(), col.data_ptr(), rows.data_ptr(), num_parts, num_nodes,
                static_cast<int64_t>(part_ptr._version()), static_cast<int64_t>(col._version()),
                static_cast<int64_t>(rows._version()), dc, Key(part_ptr), Key(col), Key(rows), Tensor(), nullptr};
    const size_t bytes = eppgcn_plan_bytes(num_parts, num_slots, num_nodes);
    void* base = nullptr;
    e.plan = aligned_bytes(bytes, part_ptr, &base);
    e.plan_ptr = base;
    const size_t wbytes = eppgcn_plan_workspace_bytes(num_parts, num_slots);
    void* wbase = nullptr;
    auto ws = aligned_bytes(wbytes, part_ptr, &wbase);
    check(eppgcn_build_plan(part_ptr.data_ptr<int32_t>(), col.data_ptr<int32_t>(),
                            is_forward ? rows.data_ptr<int32_t>() : nullptr,
                            is_forward ? nullptr : rows.data_ptr<int32_t>(), static_cast<int>(num_parts), num_slots,
                            num_nodes, dim_of_class(dc), block_shift, base, bytes, wbase, wbytes, stream_of(part_ptr)),
          "build_plan");
    // once per group array: wait for the build, refuse a plan whose look-back scan stalled and let the
    // library read the counts of the plan's stream form
    check(eppgcn_plan_status(base, static_cast<int>(num_parts), num_slots, num_nodes, nullptr, stream_of(part_ptr)),
          "build_plan");
    g_plans.push_front(std::move(e));
    trim_plans();
    return g_plans.front().plan_ptr;
}

// Per backward path, remembered from its first use:
//   - whether its plan is column-blocked: a heavily pruned path gathers from few distinct rows, which
//     stay cached in any order, so only paths that keep at least half of the edges are blocked;
//   - the bitmap of the rows it gathers, when they are fewer than half of the vertices: the
//     pre-scaling pass of the gradient then touches those rows only.
// An entry is valid for exactly the tensors it was made from (same storage, same version counters);
// see Key for why their memory cannot be handed to other tensors meanwhile.
struct PathChoice {
    const void* part_ptr;
    const void* edge_ptr;
    int64_t num_parts, num_nodes;
    int64_t version_part, version_edge;
    bool use_plan;
    Key keep_part, keep_edge;
    Tensor gathered;                           // undefined when the path reads most rows
    size_t bytes() const { return keep_part.bytes() + keep_edge.bytes() + held_bytes(gathered); }
    bool alive() const { return keep_part.alive() && keep_edge.alive(); }
    void let_go() { keep_part.held.reset(), keep_edge.held.reset(); }
};
std::list<PathChoice> g_path_choices;

const PathChoice& path_choice(const Tensor& part_pointer, const Tensor& edge_list, int64_t num_parts, int num_nodes,
                              int64_t* valid_len_out)
{
    *valid_len_out = -1;
    for (auto it = g_path_choices.begin(); it != g_path_choices.end(); ++it) {
        if (it->part_ptr == part_pointer.data_ptr() && it->edge_ptr == edge_list.data_ptr() &&
            it->num_parts == num_parts && it->num_nodes == num_nodes &&
            it->version_part == static_cast<int64_t>(part_pointer._version()) &&
            it->version_edge == static_cast<int64_t>(edge_list._version()) && it->alive()) {
            if (it != g_path_choices.begin()) {
                it->keep_part.held = part_pointer, it->keep_edge.held = edge_list;
                g_path_choices.splice(g_path_choices.begin(), g_path_choices, it);
                if (g_path_choices.size() > kAlwaysKept) std::next(g_path_choices.begin(), kAlwaysKept)->let_go();
            }
            return g_path_choices.front();
        }
    }
    const int64_t valid_len = part_pointer[num_parts].item<int64_t>();
    *valid_len_out = valid_len;
    TORCH_CHECK(valid_len >= 0 && valid_len <= edge_list.numel(), "partPointer[numParts] lies outside edgeList");
    PathChoice c{part_pointer.data_ptr(), edge_list.data_ptr(), num_parts, num_nodes,
                 static_cast<int64_t>(part_pointer._version()), static_cast<int64_t>(edge_list._version()),
                 g_plan_policy > 0 || 2 * valid_len >= edge_list.numel(), Key(part_pointer), Key(edge_list), Tensor()};
    auto bitmap = torch::empty({(static_cast<int64_t>(num_nodes) + 31) / 32 + 1}, edge_list.options());
    int64_t distinct = 0;
    const size_t scratch_bytes = eppgcn_mark_gathered_rows_scratch_bytes(num_nodes);
    auto scratch = workspace(scratch_bytes, edge_list);
    check(eppgcn_mark_gathered_rows_scratch(i32(edge_list), valid_len, num_nodes,
                                            reinterpret_cast<uint32_t*>(bitmap.data_ptr<int32_t>()),
                                            bitmap.data_ptr<int32_t>() + bitmap.numel() - 1, &distinct, scratch.data_ptr(),
                                            scratch_bytes, stream_of(edge_list)),
          "mark_gathered_rows");
    if (2 * distinct < num_nodes) c.gathered = bitmap;
    g_path_choices.push_front(std::move(c));
    trim(g_path_choices, [](const PathChoice&) {});
    return g_path_choices.front();
}

// room for the pre-scaled table and, behind it, the partial sums of a call through the plan's stream form
Tensor feature_scratch(const Tensor& feats, const void* plan)
{
    const size_t n = eppgcn_plan_workspace_floats(plan, feats.size(0), static_cast<int>(feats.size(1)));
    return torch::empty({static_cast<int64_t>(n)}, feats.options());
}

// ---------------------------------------------------------------- dense update helpers
// The three products around the aggregation run in the library's tall-and-skinny kernels when the
// shapes fit them (eppgcn_update_supported) and in torch::mm otherwise; g_dense_policy -1 forces mm.
int g_dense_policy = 0;

int dense_support(const Tensor& X, const Tensor& W)
{
    if (g_dense_policy < 0) return 0;
    return eppgcn_update_supported(static_cast<int>(X.size(1)), static_cast<int>(W.size(1)));
}

// g_masked_update: 1 (default) lets the pruned backward hand the bitmap of the rows it wrote to the dense products
// (rows outside the path are then neither cleared nor read); 0 clears and reads every row.
int g_masked_update = 1;

// {dX or an empty tensor, dW} from the aggregated gradient G; `rows`: nullptr, or the bitmap of the rows of G that
// are defined (the others count as zeros and are not read)
std::vector<Tensor> dense_backward(const Tensor& G, const Tensor& X, const Tensor& W, bool need_dx, bool relu_input,
                                   const uint32_t* rows = nullptr)
{
    const int64_t n = X.size(0);
    const int in_dim = static_cast<int>(X.size(1)), out_dim = static_cast<int>(W.size(1));
    const int sup = dense_support(X, W);
    Tensor d_weight, d_input;
    if (rows) {
        // only reached when the shapes fit the library's kernels (the caller checked dense_support)
        d_weight = torch::empty({in_dim, out_dim}, X.options());
        d_input = need_dx ? torch::empty({n, in_dim}, X.options()) : torch::empty({0}, X.options());
        const size_t nbytes = eppgcn_update_workspace_bytes(n, in_dim, out_dim);
        auto ws = torch::empty({static_cast<int64_t>((nbytes + 3) / 4) + 1}, X.options());
        check(eppgcn_update_backward_rows(need_dx ? d_input.data_ptr<float>() : nullptr, d_weight.data_ptr<float>(), f32(X),
                                          f32(G), f32(W), relu_input ? 1 : 0, rows, n, in_dim, out_dim,
                                          ws.data_ptr<float>(), nbytes, stream_of(X)),
              "update_backward_rows");
        return {d_input, d_weight};
    }
    if (need_dx && (sup & 6) == 6) {
        // both gradients from one call: narrow layers read X and G once for the two products
        d_weight = torch::empty({in_dim, out_dim}, X.options());
        d_input = torch::empty({n, in_dim}, X.options());
        const size_t nbytes = eppgcn_update_workspace_bytes(n, in_dim, out_dim);
        auto ws = torch::empty({static_cast<int64_t>((nbytes + 3) / 4) + 1}, X.options());
        check(eppgcn_update_backward(d_input.data_ptr<float>(), d_weight.data_ptr<float>(), f32(X), f32(G), f32(W),
                                     relu_input ? 1 : 0, n, in_dim, out_dim, ws.data_ptr<float>(), nbytes, stream_of(X)),
              "update_backward");
        return {d_input, d_weight};
    }
    if (sup & 4) {
        d_weight = torch::empty({in_dim, out_dim}, X.options());
        const size_t nbytes = eppgcn_update_workspace_bytes(n, in_dim, out_dim);
        auto ws = torch::empty({static_cast<int64_t>((nbytes + 3) / 4) + 1}, X.options());
        check(eppgcn_update_backward_weight(d_weight.data_ptr<float>(), f32(X), f32(G), relu_input ? 1 : 0, n, in_dim,
                                            out_dim, ws.data_ptr<float>(), nbytes, stream_of(X)),
              "update_backward_weight");
    } else {
        d_weight = torch::mm((relu_input ? torch::relu(X) : X).transpose(0, 1), G);
    }
    if (!need_dx) {
        d_input = torch::empty({0}, X.options());
    } else if (sup & 2) {
        d_input = torch::empty({n, in_dim}, X.options());
        check(eppgcn_update_backward_input(d_input.data_ptr<float>(), f32(G), f32(W), relu_input ? f32(X) : nullptr, n,
                                           in_dim, out_dim, stream_of(X)),
              "update_backward_input");
    } else {
        d_input = torch::mm(G, W.transpose(0, 1));
        if (relu_input) d_input = d_input * (X > 0);
    }
    return {d_input, d_weight};
}

// ---------------------------------------------------------------- forward / backward
std::vector<Tensor> forward(Tensor input, Tensor weight, Tensor row_pointers, Tensor column_index, Tensor degrees,
                            Tensor part_pointers, Tensor part2Node, int partSize, int dimWorker, int warpPerBlock,
                            bool relu_input)
{
    CHECK_F32(input); CHECK_F32(weight); CHECK_I32(row_pointers); CHECK_I32(column_index);
    CHECK_F32(degrees); CHECK_I32(part_pointers); CHECK_I32(part2Node);
    TORCH_CHECK(input.dim() == 2 && weight.dim() == 2 && input.size(1) == weight.size(0), "shape mismatch");
    TORCH_CHECK(degrees.numel() == input.size(0), "degrees must have one entry per vertex");
    TORCH_CHECK(part_pointers.numel() >= part2Node.numel() + 1, "part_pointers needs num_parts + 1 entries");
    CHECK_COUNTS(column_index, input.size(0));
    const int64_t n = input.size(0);
    const int dim = static_cast<int>(weight.size(1));
    auto output = torch::empty({n, dim}, input.options());
    const void* plan = plan_for(part_pointers, column_index, part2Node, true, part2Node.numel(), column_index.numel(),
                                static_cast<int>(n), dim);
    if (n > 0 && (dense_support(input, weight) & 1)) {
        // the product is written scaled and padded, ready to be gathered: no separate scaling pass
        const size_t ws_floats = eppgcn_plan_workspace_floats(plan, n, dim);
        auto scaled = torch::empty({static_cast<int64_t>(ws_floats)}, input.options());
        check(eppgcn_layer_forward(output.data_ptr<float>(), input.data_ptr<float>(), weight.data_ptr<float>(), relu_input ? 1 : 0,
                                   i32(row_pointers), i32(column_index), f32(degrees), i32(part_pointers), i32(part2Node),
                                   static_cast<int>(n), static_cast<int>(input.size(1)), dim,
                                   static_cast<int>(part2Node.numel()), partSize, dimWorker, warpPerBlock,
                                   scaled.data_ptr<float>(), ws_floats, plan, stream_of(input)),
              "forward");
        return {output};
    }
    auto tmp = torch::mm(relu_input ? torch::relu(input) : input, weight);
    // tmp is ours: when its rows need no padding and no partial sums follow the table it is scaled in place,
    // otherwise into scratch
    const size_t ws_floats = eppgcn_plan_workspace_floats(plan, tmp.size(0), dim);
    auto scaled = ws_floats == static_cast<size_t>(tmp.numel())
                      ? tmp
                      : torch::empty({static_cast<int64_t>(ws_floats)}, tmp.options());
    check(eppgcn_spmm_forward(output.data_ptr<float>(), f32(tmp), i32(row_pointers), i32(column_index),
                              f32(degrees), i32(part_pointers), i32(part2Node), static_cast<int>(n), dim,
                              static_cast<int>(part2Node.numel()), partSize, dimWorker, warpPerBlock,
                              scaled.numel() ? scaled.data_ptr<float>() : nullptr, ws_floats, plan, stream_of(input)),
          "forward");
    return {output};
}

std::vector<Tensor> backward(Tensor d_output, Tensor X, Tensor W, Tensor row_pointers, Tensor column_index,
                             Tensor degrees, Tensor part_pointers, Tensor part2Node, int partSize, int dimWorker,
                             int warpPerBlock, bool need_dx, bool relu_input)
{
    CHECK_F32(d_output); CHECK_F32(X); CHECK_F32(W); CHECK_I32(row_pointers); CHECK_I32(column_index);
    CHECK_F32(degrees); CHECK_I32(part_pointers); CHECK_I32(part2Node);
    TORCH_CHECK(d_output.dim() == 2 && degrees.numel() == d_output.size(0), "shape mismatch");
    TORCH_CHECK(X.dim() == 2 && W.dim() == 2 && X.size(0) == d_output.size(0) && X.size(1) == W.size(0) &&
                    W.size(1) == d_output.size(1), "X, W and d_output do not fit together");
    TORCH_CHECK(part_pointers.numel() >= part2Node.numel() + 1, "part_pointers needs num_parts + 1 entries");
    CHECK_COUNTS(column_index, d_output.size(0));
    auto d_input_prime = torch::empty_like(d_output);
    const void* plan = plan_for(part_pointers, column_index, part2Node, true, part2Node.numel(), column_index.numel(),
                                static_cast<int>(d_output.size(0)), static_cast<int>(d_output.size(1)));
    auto scaled = feature_scratch(d_output, plan);     // d_output belongs to autograd: scale into scratch
    check(eppgcn_spmm_backward(d_input_prime.data_ptr<float>(), f32(d_output), i32(row_pointers),
                               i32(column_index), f32(degrees), i32(part_pointers), i32(part2Node),
                               static_cast<int>(d_output.size(0)), static_cast<int>(d_output.size(1)),
                               static_cast<int>(part2Node.numel()), partSize, dimWorker, warpPerBlock,
                               scaled.numel() ? scaled.data_ptr<float>() : nullptr, static_cast<size_t>(scaled.numel()),
                               plan, stream_of(d_output)),
          "backward");
    return dense_backward(d_input_prime, X, W, need_dx, relu_input);
}

void mask_forward(Tensor id, Tensor partPointer, Tensor edgeList, Tensor src_mask, Tensor ngh_mask,
                  Tensor backEdgeMask, Tensor node_degs, int num_layers, int layer, int blockx, int blocky)
{
    CHECK_I32(id); CHECK_I32(partPointer); CHECK_I32(edgeList); CHECK_MASK(src_mask); CHECK_MASK(ngh_mask);
    CHECK_I32(backEdgeMask); CHECK_I32(node_degs);
    const bool is_last = layer == num_layers;
    TORCH_CHECK(partPointer.numel() >= id.numel() + 1, "partPointer needs num_parts + 1 entries");
    TORCH_CHECK(backEdgeMask.numel() >= edgeList.numel(), "backEdgeMask is shorter than the edge list");
    TORCH_CHECK(src_mask.numel() == node_degs.numel(), "src_mask and node_degs must have one entry per vertex");
    CHECK_COUNTS(edgeList, node_degs.numel());
    TORCH_CHECK(is_last || ngh_mask.numel() == node_degs.numel(), "ngh_mask must have one entry per vertex");
    check(eppgcn_mask_forward(i32(id), i32(partPointer), i32(edgeList),
                              static_cast<const uint8_t*>(src_mask.data_ptr()),
                              ngh_mask.numel() ? static_cast<uint8_t*>(ngh_mask.data_ptr()) : nullptr,
                              backEdgeMask.data_ptr<int32_t>(), node_degs.data_ptr<int32_t>(),
                              static_cast<int>(id.numel()), edgeList.numel(), is_last ? 1 : 0, blockx, blocky,
                              stream_of(id)),
          "mask_forward");
}

std::vector<Tensor> ours_backward(Tensor d_output, Tensor X, Tensor W, Tensor id, Tensor partPointer, Tensor edgeList,
                                  Tensor degrees, int partSize, int numParts, int layer, int blockx, int blocky,
                                  bool need_dx, bool relu_input)
{
    CHECK_F32(d_output); CHECK_F32(X); CHECK_F32(W); CHECK_I32(id); CHECK_I32(partPointer); CHECK_I32(edgeList);
    CHECK_F32(degrees);
    TORCH_CHECK(d_output.dim() == 2 && degrees.numel() == d_output.size(0), "shape mismatch");
    TORCH_CHECK(X.dim() == 2 && W.dim() == 2 && X.size(0) == d_output.size(0) && X.size(1) == W.size(0) &&
                    W.size(1) == d_output.size(1), "X, W and d_output do not fit together");
    TORCH_CHECK(numParts >= 0 && partPointer.numel() >= static_cast<int64_t>(numParts) + 1,
                "partPointer needs numParts + 1 entries");
    CHECK_COUNTS(edgeList, d_output.size(0));
    auto d_input_prime = torch::empty_like(d_output);
    const int num_nodes = static_cast<int>(d_output.size(0));
    const void* plan = nullptr;
    const uint32_t* gathered = nullptr;
    if (numParts > 0) {
        int64_t valid_len = -1;
        const PathChoice& choice = path_choice(partPointer, edgeList, numParts, num_nodes, &valid_len);
        if (choice.gathered.defined())
            gathered = reinterpret_cast<const uint32_t*>(choice.gathered.data_ptr<int32_t>());
        // a heavily pruned path keeps its groups in one block (its few gathered rows stay cached anyway)
        plan = plan_for(partPointer, edgeList, id, false, numParts, valid_len, num_nodes,
                        static_cast<int>(d_output.size(1)), choice.use_plan ? 0 : 31);
    }
    auto scaled = feature_scratch(d_output, plan);     // d_output belongs to autograd: scale into scratch
    // The aggregated gradient is only read by the two dense products below.  When they run in the library's kernels
    // (which take the bitmap of the rows the aggregation wrote), the rows outside the path are neither cleared
    // nor read - the row-masked products the reference sketches in its comments (EPPGCN_kernel.cu:607,616).
    const int sup = dense_support(X, W);
    const bool masked = g_masked_update > 0 && plan && (sup & 4) && (!need_dx || (sup & 2));
    const uint32_t* written = nullptr;
    if (masked) {
        check(eppgcn_ours_backward_rows(d_input_prime.data_ptr<float>(), f32(d_output), i32(id), i32(partPointer),
                                        i32(edgeList), f32(degrees), static_cast<int>(d_output.size(0)),
                                        static_cast<int>(d_output.size(1)), numParts, partSize > 0 ? partSize : 1, layer,
                                        blockx, blocky, scaled.numel() ? scaled.data_ptr<float>() : nullptr,
                                        static_cast<size_t>(scaled.numel()), plan, gathered, &written, nullptr,
                                        stream_of(d_output)),
              "ours_backward_rows");
    } else {
        check(eppgcn_ours_backward(d_input_prime.data_ptr<float>(), f32(d_output), i32(id), i32(partPointer),
                                   i32(edgeList), f32(degrees), static_cast<int>(d_output.size(0)),
                                   static_cast<int>(d_output.size(1)), numParts, partSize > 0 ? partSize : 1, layer, blockx,
                                   blocky, scaled.numel() ? scaled.data_ptr<float>() : nullptr,
                                   static_cast<size_t>(scaled.numel()), plan, gathered, stream_of(d_output)),
              "ours_backward");
    }
    return dense_backward(d_input_prime, X, W, need_dx, relu_input, written);
}

// ---------------------------------------------------------------- training loss
// rows: int64 ids of the training rows; labels: class of every vertex, -1 outside the training rows
Tensor nll_forward(Tensor logits, Tensor rows, Tensor labels)
{
    CHECK_F32(logits); CHECK_INPUT(rows); CHECK_I32(labels);
    TORCH_CHECK(rows.scalar_type() == torch::kInt64, "rows must be int64");
    TORCH_CHECK(logits.dim() == 2 && labels.numel() == logits.size(0), "labels must have one entry per row of logits");
    auto loss = torch::empty({}, logits.options());
    const size_t nbytes = eppgcn_nll_workspace_bytes();
    auto ws = workspace(nbytes, logits);
    check(eppgcn_nll_forward(loss.data_ptr<float>(), f32(logits), rows.numel() ? rows.data_ptr<int64_t>() : nullptr, i32(labels),
                             rows.numel(), logits.size(0), static_cast<int>(logits.size(1)), ws.data_ptr(), nbytes,
                             stream_of(logits)),
          "nll_forward");
    return loss;
}

Tensor nll_backward(Tensor d_loss, Tensor logits, Tensor labels, int64_t num_rows)
{
    CHECK_F32(d_loss); CHECK_F32(logits); CHECK_I32(labels);
    TORCH_CHECK(d_loss.numel() == 1, "d_loss must be one number");
    TORCH_CHECK(logits.dim() == 2 && labels.numel() == logits.size(0), "labels must have one entry per row of logits");
    auto grad = torch::empty_like(logits);
    check(eppgcn_nll_backward(grad.numel() ? grad.data_ptr<float>() : nullptr, d_loss.data_ptr<float>(), f32(logits), i32(labels),
                              num_rows, logits.size(0), static_cast<int>(logits.size(1)), stream_of(logits)),
          "nll_backward");
    return grad;
}

// ---------------------------------------------------------------- autograd functions in native code
// What gcn_conv.GNNAFunction and train._TrainingLoss do, without the Python calls in both directions (the backward ones run on
// the engine's thread, which has to get the interpreter for each).  They are for plain tensors in ordinary eager autograd; for
// anything that looks into or changes how functions run - function transforms, forward-mode gradients, dispatch and function
// modes, tracing, profiling, subclasses - the callers take the Python functions, which behave as torch defines it for those.
// A small graph's epoch is bound by the host that issues its 17 launches: 216-240 us at 2 708 vertices with the Python functions over
// eight processes, 177-189 with these, the kept unit gradient and drop_gradients below in place of torch's own (single processes
// 215, these alone 181, all 163); its kernels take 66.
bool plain_eager(std::initializer_list<const Tensor*> tensors)
{
    using c10::DispatchKey;
    if (c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled() || at::hasCallbacks()) return false;
    if (c10::impl::tls_local_dispatch_key_set().included_.has_any(
            c10::DispatchKeySet({DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::Tracer, DispatchKey::Python})))
        return false;
    const c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                       DispatchKey::Functionalize, DispatchKey::Negative, DispatchKey::Conjugate});
    for (const Tensor* t : tensors) {
        if (!t->defined() || t->layout() != torch::kStrided || !t->is_cuda() || t->key_set().has_any(wrapped) || t->is_inference())
            return false;
        if (t->_fw_grad(0).defined()) return false;
    }
    return true;
}

// An attribute of a record, with the error that the Python function's call of the module gives for one of another type.
template <class T>
T value_of(const pybind11::object& value, const char* name)
{
    try {
        return value.cast<T>();
    } catch (const pybind11::cast_error&) {
        PyErr_Format(PyExc_TypeError, "%s of the layer's record has a type that the operation does not take", name);
        throw pybind11::error_already_set();
    }
}
template <class T>
T arg_of(const pybind11::object& record, const char* name)
{
    return value_of<T>(record.attr(name), name);
}

// What the Python functions keep on ctx, which a caller finds - and can set - on a result's grad_fn, and which the backward pass
// reads when it runs: a layer's backward path is filled in after its first forward pass.  It becomes a dict when somebody looks
// (made in each pass, an epoch of 2 708 vertices took 175 us for 170).  A node holds it by the storage of a one-element tensor,
// since that is a kind of saved data that compiled autograd can hand on; the element is its own address, so that a copy of the
// tensor is recognised.
struct Attributes {
    enum Kind { kObject, kNumber, kTruth };
    struct Name {
        const char* name;
        Kind kind;
        int at;                                          // in objects (an object) or numbers (the others)
    };
    int64_t address;
    const Name* names;
    int count;
    pybind11::object objects[2];                         // the values until there is a dict
    int64_t numbers[4];
    pybind11::object dict;
    static Tensor held(Attributes* a)
    {
        a->address = reinterpret_cast<int64_t>(a);
        return torch::from_blob(&a->address, {1}, [a](void*) { let_go(a); }, torch::kInt64);
    }
    static Attributes& of(const Tensor& held)
    {
        const int64_t* at = held.data_ptr<int64_t>();
        TORCH_CHECK(*at == reinterpret_cast<int64_t>(at), "the function's attributes were copied");
        return *reinterpret_cast<Attributes*>(*at);
    }
    pybind11::dict as_dict()
    {
        if (!dict) {
            pybind11::dict made;
            for (int k = 0; k < count; ++k) {
                const Name& n = names[k];
                if (n.kind == kObject) made[n.name] = objects[n.at];
                else if (n.kind == kTruth) made[n.name] = pybind11::bool_(numbers[n.at] != 0);
                else made[n.name] = pybind11::int_(numbers[n.at]);
            }
            dict = std::move(made);
            for (auto& value : objects) value = pybind11::object();
        }
        return pybind11::reinterpret_borrow<pybind11::dict>(dict);
    }
    pybind11::object in_dict(int k) const
    {
        PyObject* value = PyDict_GetItemString(dict.ptr(), names[k].name);
        if (!value) {
            PyErr_Format(PyExc_AttributeError, "the function has no attribute '%s'", names[k].name);
            throw pybind11::error_already_set();
        }
        return pybind11::reinterpret_borrow<pybind11::object>(value);
    }
    pybind11::object object(int k) const { return dict ? in_dict(k) : objects[names[k].at]; }
    template <class T>
    T number(int k) const
    {
        return dict ? value_of<T>(in_dict(k), names[k].name) : static_cast<T>(numbers[names[k].at]);
    }
    static void let_go(Attributes* a)
    {
        if (!Py_IsInitialized()) return;                 // nothing is left to give the objects back to
        pybind11::gil_scoped_acquire gil;
        delete a;
    }
};
static_assert(offsetof(Attributes, address) == 0, "the element's address is the object's");

// grad_fn of a native function F with kInputs inputs: the saved tensors, the inputs that need gradients, and the attributes above.
template <class F, int kInputs>
struct NodeType {
    using Node = torch::autograd::CppNode<F>;
    static PyTypeObject type;
    static Node& node(PyObject* self)
    {
        return dynamic_cast<Node&>(*reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata);
    }
    static pybind11::dict attributes(PyObject* self)
    {
        return F::attributes(node(self).ctx_).as_dict();
    }
    static PyObject* get(PyObject* self, PyObject* name)
    {
        HANDLE_TH_ERRORS
        PyObject* found = PyObject_GenericGetAttr(self, name);
        if (found || !PyErr_ExceptionMatches(PyExc_AttributeError)) return found;
        pybind11::error_already_set missing;
        PyObject* value = PyDict_GetItemWithError(attributes(self).ptr(), name);
        if (!value && !PyErr_Occurred()) missing.restore();
        Py_XINCREF(value);
        return value;
        END_HANDLE_TH_ERRORS
    }
    static int set(PyObject* self, PyObject* name, PyObject* value)
    {
        HANDLE_TH_ERRORS
        if (PyObject_HasAttr(reinterpret_cast<PyObject*>(&type), name)) return PyObject_GenericSetAttr(self, name, value);
        const pybind11::dict values = attributes(self);
        if (value) return PyObject_SetItem(values.ptr(), name, value);
        if (PyDict_Contains(values.ptr(), name) == 0) {
            PyErr_SetObject(PyExc_AttributeError, name);
            return -1;
        }
        return PyObject_DelItem(values.ptr(), name);
        END_HANDLE_TH_ERRORS_RET(-1)
    }
    static PyObject* dict(PyObject* self, void*)
    {
        HANDLE_TH_ERRORS
        return attributes(self).release().ptr();
        END_HANDLE_TH_ERRORS
    }
    static PyObject* saved_tensors(PyObject* self, void*)
    {
        HANDLE_TH_ERRORS
        return pybind11::tuple(pybind11::cast(node(self).ctx_.get_saved_variables())).release().ptr();
        END_HANDLE_TH_ERRORS
    }
    static PyObject* needs_input_grad(PyObject* self, void*)
    {
        HANDLE_TH_ERRORS
        const Node& n = node(self);
        pybind11::tuple needs(kInputs);
        for (uint32_t k = 0; k < kInputs; ++k) needs[k] = pybind11::bool_(k < n.num_outputs() && n.next_edge(k).is_valid());
        return needs.release().ptr();
        END_HANDLE_TH_ERRORS
    }
    static void add(const char* name)
    {
        using namespace torch::autograd;                 // for the names in the macro
        if (type.tp_flags & Py_TPFLAGS_READY) return;    // the module is imported under a second name
        static PyGetSetDef properties[] = {THP_FUNCTION_DEFAULT_PROPERTIES,
                                           {"saved_tensors", saved_tensors, nullptr, nullptr, nullptr},
                                           {"needs_input_grad", needs_input_grad, nullptr, nullptr, nullptr},
                                           {"__dict__", dict, nullptr, nullptr, nullptr},
                                           {nullptr}};
        type.tp_getattro = get;
        type.tp_setattro = set;
        _initFunctionPyTypeObject(type, name, properties, nullptr);
        registerCppFunction(typeid(Node), &type);
        Py_INCREF(&type);                                // it is never freed
        const auto added = pybind11::reinterpret_borrow<pybind11::object>(reinterpret_cast<PyObject*>(&type));
        pybind11::module_::import("torch.autograd.graph").attr("Node").attr("register")(added);      // isinstance, as for Python's
    }
};
template <class F, int kInputs>
PyTypeObject NodeType<F, kInputs>::type{};

struct GraphArgs {
    Tensor row_pointers, column_index, degrees, part_ptr, part2node;
    int part_size, dim_worker, warp_per_block;
    explicit GraphArgs(const pybind11::object& info)
        : row_pointers(arg_of<Tensor>(info, "row_pointers")), column_index(arg_of<Tensor>(info, "column_index")),
          degrees(arg_of<Tensor>(info, "degrees")), part_ptr(arg_of<Tensor>(info, "partPtr")),
          part2node(arg_of<Tensor>(info, "part2Node")), part_size(arg_of<int>(info, "partSize")),
          dim_worker(arg_of<int>(info, "dimWorker")), warp_per_block(arg_of<int>(info, "warpPerBlock")) {}
};

struct PathArgs {
    Tensor id, part_pointer, edge_list, degrees;
    int part_size, num_parts, layer, blockx, blocky;
    explicit PathArgs(const pybind11::object& back)
        : id(arg_of<Tensor>(back, "id")), part_pointer(arg_of<Tensor>(back, "partPointer")),
          edge_list(arg_of<Tensor>(back, "edgeList")), degrees(arg_of<Tensor>(back, "degrees")),
          part_size(arg_of<int>(back, "partSize")), num_parts(arg_of<int>(back, "numParts")),
          layer(arg_of<int>(back, "layer")), blockx(arg_of<int>(back, "blockx")), blocky(arg_of<int>(back, "blocky")) {}
};

struct GNNAFunction : torch::autograd::Function<GNNAFunction> {
    enum { kInfo, kBack, kRelu };
    static constexpr Attributes::Name kNames[] = {
        {"inputInfo", Attributes::kObject, 0}, {"backInfo", Attributes::kObject, 1}, {"reluInput", Attributes::kTruth, 0},
        {"partSize", Attributes::kNumber, 1}, {"dimWorker", Attributes::kNumber, 2}, {"warpPerBlock", Attributes::kNumber, 3}};
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& X, const Tensor& W,
                          const pybind11::object& info, const pybind11::object& back, bool relu_input)
    {
        ctx->save_for_backward({X, W});
        const GraphArgs g(info);
        ctx->saved_data["attributes"] = Attributes::held(new Attributes{
            0, kNames, 6, {info, back}, {relu_input, g.part_size, g.dim_worker, g.warp_per_block}, {}});
        return ::forward(X, W, g.row_pointers, g.column_index, g.degrees, g.part_ptr, g.part2node, g.part_size, g.dim_worker,
                         g.warp_per_block, relu_input)[0];
    }
    static Attributes& attributes(torch::autograd::AutogradContext& ctx)
    {
        return Attributes::of(ctx.saved_data.at("attributes").toTensor());
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &X = saved[0], &W = saved[1], d_output = grads[0].contiguous();
        const bool need_dx = ctx->needs_input_grad(0);
        std::vector<Tensor> d;
        pybind11::gil_scoped_acquire gil;                // for the records, and for the caches above as in every other call
        const Attributes& kept = attributes(*ctx);
        const pybind11::object back = kept.object(kBack);
        const bool relu_input = kept.number<bool>(kRelu);
        const pybind11::object unpruned = pybind11::getattr(back, "unpruned", pybind11::none());
        const int all_edges = PyObject_IsTrue(unpruned.ptr());
        if (all_edges < 0) throw pybind11::error_already_set();
        if (all_edges) {
            const GraphArgs g(kept.object(kInfo));
            d = ::backward(d_output, X, W, g.row_pointers, g.column_index, g.degrees, g.part_ptr, g.part2node, g.part_size,
                           g.dim_worker, g.warp_per_block, need_dx, relu_input);
        } else {
            const PathArgs p(back);
            d = ours_backward(d_output, X, W, p.id, p.part_pointer, p.edge_list, p.degrees, p.part_size, p.num_parts, p.layer,
                              p.blockx, p.blocky, need_dx, relu_input);
        }
        return {need_dx ? d[0] : Tensor(), d[1], Tensor(), Tensor(), Tensor()};
    }
};
using GNNAFunctionBackward = NodeType<GNNAFunction, 8>;      // the Python function takes eight inputs

// The layer's forward pass with the autograd function above; nullopt: the caller takes the Python function.
std::optional<Tensor> gcn_layer(const Tensor& X, const Tensor& W, pybind11::object info, pybind11::object back, bool relu_input)
{
    if (!plain_eager({&X, &W})) return std::nullopt;
    return GNNAFunction::apply(X, W, info, back, relu_input);
}

struct TrainingLoss : torch::autograd::Function<TrainingLoss> {
    static constexpr Attributes::Name kNames[] = {{"num_rows", Attributes::kNumber, 0}};
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& logits, const Tensor& rows, const Tensor& labels)
    {
        ctx->save_for_backward({logits, labels});
        ctx->saved_data["num_rows"] = rows.numel();
        return nll_forward(logits, rows, labels);
    }
    static Attributes& attributes(torch::autograd::AutogradContext& ctx)
    {
        auto& held = ctx.saved_data["attributes"];
        if (!held.isTensor()) held = Attributes::held(new Attributes{0, kNames, 1, {}, {ctx.saved_data.at("num_rows").toInt()}, {}});
        return Attributes::of(held.toTensor());
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const bool twice = torch::GradMode::is_enabled() && grads[0].requires_grad();
        const bool looked_at = ctx->saved_data.find("attributes") != ctx->saved_data.end();
        Tensor d;
        {
            torch::NoGradGuard no_grad;
            pybind11::gil_scoped_acquire gil;            // one call into the library at a time, as from Python
            const int64_t num_rows = looked_at ? attributes(*ctx).number<int64_t>(0) : ctx->saved_data["num_rows"].toInt();
            d = nll_backward(grads[0].contiguous(), saved[0], saved[1], num_rows);
        }
        if (twice) {                                     // as Python's once_differentiable: an error if it is differentiated
            auto error = std::make_shared<torch::autograd::DelayedError>(
                "trying to differentiate twice a function that was marked with @once_differentiable", 1);
            d = error->apply({d.detach().set_requires_grad(true)})[0];
        }
        return {d, Tensor(), Tensor()};
    }
};

using TrainingLossBackward = NodeType<TrainingLoss, 3>;

std::optional<Tensor> training_loss(const Tensor& logits, const Tensor& rows, const Tensor& labels)
{
    if (!plain_eager({&logits, &rows, &labels})) return std::nullopt;
    return TrainingLoss::apply(logits, rows, labels);
}

// A loss that is training_loss's own result, with no hook on its node: its backward pass starts in the library, which only reads
// the gradient it is given, and nobody else is handed it.
bool gradient_stays_unseen(const Tensor& loss)
{
    const auto node = loss.defined() ? loss.grad_fn() : nullptr;
    return dynamic_cast<TrainingLossBackward::Node*>(node.get()) && node->pre_hooks().empty() &&
           node->tensor_pre_hooks().empty() && node->post_hooks().empty();
}

// ---------------------------------------------------------------- optimizer
// One Adam step of all weights in one launch, in the rounding of torch's grouped operations; `steps` are the optimizer's CPU
// counters.  False, with nothing changed, for weights, gradients or state of another form than fp32, contiguous and on one
// GPU, for beta1 <= 0.5 (torch then rounds its average another way) and under graph capture (where torch's Adam asks for its
// capturable form): the caller then takes torch's step.
bool adam_step(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& exp_avg,
               const std::vector<Tensor>& exp_avg_sq, const std::vector<Tensor>& steps, double lr, double beta1, double beta2,
               double eps)
{
    const size_t count = params.size();
    if (count == 0 || grads.size() != count || exp_avg.size() != count || exp_avg_sq.size() != count || steps.size() != count)
        return false;
    if (!(beta1 > 0.5 && beta1 < 1.0 && beta2 >= 0.0 && beta2 < 1.0)) return false;
    const auto device = params[0].device();
    const auto plain = [&](const Tensor& t, const Tensor& p) {
        return t.defined() && t.layout() == torch::kStrided && t.is_cuda() && t.device() == device &&
               t.scalar_type() == torch::kFloat32 && t.is_contiguous() && t.sizes() == p.sizes() && !t.is_inference();
    };
    for (size_t k = 0; k < count; ++k) {
        const Tensor& s = steps[k];
        if (!plain(params[k], params[k]) || !plain(grads[k], params[k]) || !plain(exp_avg[k], params[k]) ||
            !plain(exp_avg_sq[k], params[k]))
            return false;
        if (!s.defined() || s.layout() != torch::kStrided || !s.is_cpu() || s.scalar_type() != torch::kFloat32 ||
            s.numel() != 1 || s.is_inference())
            return false;
        if (!(s.data_ptr<float>()[0] >= 0.f && s.data_ptr<float>()[0] < 16777215.f)) return false;
    }
    if (device.index() != c10::hip::current_device()) return false;
    if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return false;
    RECORD_USER_SCOPE("Optimizer.step#Adam.step");      // the range a profile of torch's own step has
    std::vector<float*> p(count), m(count), v(count);
    std::vector<const float*> g(count);
    std::vector<int64_t> sizes(count);
    std::vector<double> at(count);
    for (size_t k = 0; k < count; ++k) steps[k].data_ptr<float>()[0] += 1.f;      // before any is read: weights may share one
    for (size_t k = 0; k < count; ++k) {
        p[k] = params[k].data_ptr<float>(), m[k] = exp_avg[k].data_ptr<float>(), v[k] = exp_avg_sq[k].data_ptr<float>();
        g[k] = grads[k].data_ptr<float>();
        sizes[k] = params[k].numel();
        at[k] = static_cast<double>(steps[k].data_ptr<float>()[0]);
    }
    check(eppgcn_adam_step(static_cast<int>(count), p.data(), g.data(), m.data(), v.data(), sizes.data(), at.data(), lr, beta1,
                           beta2, eps, stream_of(params[0])),
          "adam_step");
    for (size_t k = 0; k < count; ++k) {
        // written behind torch's back: a graph that saved one of them has to see that it changed
        for (const Tensor* t : {&params[k], &exp_avg[k], &exp_avg_sq[k], &steps[k]}) t->unsafeGetTensorImpl()->bump_version();
    }
    return true;
}

// The gradients of these weights are given up, as torch's zero_grad does (set_to_none), with the range that a profile of it has.
void drop_gradients(const std::vector<Tensor>& params)
{
    RECORD_USER_SCOPE("Optimizer.zero_grad#Adam.zero_grad");
    for (const Tensor& p : params)
        if (p.grad().defined()) p.mutable_grad().reset();
}

// ---------------------------------------------------------------- path preparation
std::vector<Tensor> build_part(int partSize, Tensor indptr)
{
    TORCH_CHECK(partSize >= 1, "partSize must be >= 1");
    TORCH_CHECK(indptr.scalar_type() == torch::kInt32 && indptr.dim() == 1 && indptr.numel() >= 1,
                "indptr must be a 1-D int32 tensor");
    auto dptr = indptr.is_cuda() ? indptr.contiguous() : indptr.contiguous().to(torch::kCUDA);
    const int num_nodes = static_cast<int>(dptr.numel() - 1);
    const int64_t num_edges = (dptr[num_nodes] - dptr[0]).item<int64_t>();
    const int64_t capacity = num_edges / partSize + num_nodes + 1;
    auto part_ptr = torch::empty({capacity}, dptr.options());
    auto part2node = torch::empty({capacity > 1 ? capacity - 1 : 1}, dptr.options());
    const size_t bytes = eppgcn_split_workspace_bytes(num_nodes);
    auto ws = workspace(bytes, dptr);
    int64_t num_parts = 0;
    check(eppgcn_build_part(dptr.data_ptr<int32_t>(), num_nodes, partSize, part_ptr.data_ptr<int32_t>(),
                            part2node.data_ptr<int32_t>(), capacity, ws.data_ptr(), bytes, nullptr, &num_parts,
                            stream_of(dptr)),
          "build_part");
    return {part_ptr.narrow(0, 0, num_parts + 1), part2node.narrow(0, 0, num_parts)};
}

struct Compacted {
    Tensor id, edge_list;
    int64_t valid_len;
};

Compacted compact(const Tensor& edge_mask, const Tensor& column_index)
{
    CHECK_I32(edge_mask); CHECK_I32(column_index);
    TORCH_CHECK(column_index.numel() >= edge_mask.numel(), "column_index is shorter than edge_mask");
    const int64_t length = edge_mask.numel();
    Compacted c{torch::empty_like(edge_mask), torch::empty({length}, column_index.options()), 0};
    const size_t bytes = eppgcn_compact_workspace_bytes(length);
    auto ws = workspace(bytes, edge_mask);
    check(eppgcn_compact_back_edge(i32(edge_mask), i32(column_index), c.id.data_ptr<int32_t>(),
                                   c.edge_list.data_ptr<int32_t>(), length, ws.data_ptr(), bytes, nullptr,
                                   &c.valid_len, stream_of(edge_mask)),
          "compact_back_edge");
    return c;
}

int64_t valid_nodes(const Tensor& node_deg)
{
    CHECK_I32(node_deg);
    auto d = torch::empty({1}, node_deg.options());
    int64_t v = 0;
    check(eppgcn_count_nonzero(i32(node_deg), node_deg.numel(), d.data_ptr<int32_t>(), &v, stream_of(node_deg)),
          "count_nonzero");
    return v;
}

struct Split {
    Tensor part_pointer;
    int64_t num_parts;
};

Split split(const Tensor& node_deg, int64_t num_edges, int part_size)
{
    CHECK_I32(node_deg);
    TORCH_CHECK(part_size >= 1, "back_part_size must be >= 1");
    TORCH_CHECK(num_edges >= 0, "num_edges must be >= 0");
    Split s{torch::empty({num_edges + 1}, node_deg.options()), 0};
    const size_t bytes = eppgcn_split_workspace_bytes(node_deg.numel());
    auto ws = workspace(bytes, node_deg);
    check(eppgcn_split_back_part(i32(node_deg), static_cast<int>(node_deg.numel()), part_size,
                                 s.part_pointer.data_ptr<int32_t>(), num_edges + 1, ws.data_ptr(), bytes, nullptr,
                                 &s.num_parts, nullptr, stream_of(node_deg)),
          "split_back_part");
    return s;
}

std::vector<Tensor> compact_back_edge(Tensor edge_mask, Tensor column_index)
{
    auto c = compact(edge_mask, column_index);
    auto info = torch::zeros({1}, torch::kFloat64);
    info[0] = static_cast<double>(c.valid_len);
    return {c.id, c.edge_list, info};
}

// Addition: mask_forward and compact_back_edge of one layer in one pass, same arguments as
// mask_forward minus the edge mask and the launch hints; returns what compact_back_edge returns.
std::vector<Tensor> mark_compact(Tensor id, Tensor partPointer, Tensor edgeList, Tensor src_mask, Tensor ngh_mask,
                                 Tensor node_degs, int num_layers, int layer)
{
    CHECK_I32(id); CHECK_I32(partPointer); CHECK_I32(edgeList); CHECK_MASK(src_mask); CHECK_MASK(ngh_mask);
    CHECK_I32(node_degs);
    const bool is_last = layer == num_layers;
    TORCH_CHECK(partPointer.numel() >= id.numel() + 1, "partPointer needs num_parts + 1 entries");
    TORCH_CHECK(src_mask.numel() == node_degs.numel(), "src_mask and node_degs must have one entry per vertex");
    CHECK_COUNTS(edgeList, node_degs.numel());
    TORCH_CHECK(is_last || ngh_mask.numel() == node_degs.numel(), "ngh_mask must have one entry per vertex");
    const int64_t length = edgeList.numel();
    auto out_id = torch::empty({length}, edgeList.options());
    auto out_edge = torch::empty({length}, edgeList.options());
    const size_t nbytes = eppgcn_mark_compact_workspace_bytes(length);
    auto ws = torch::empty({static_cast<int64_t>((nbytes + 7) / 8)}, edgeList.options().dtype(torch::kInt64));
    int64_t valid_len = 0;
    check(eppgcn_mark_compact(i32(id), i32(partPointer), i32(edgeList), static_cast<const uint8_t*>(src_mask.data_ptr()),
                              ngh_mask.numel() ? static_cast<uint8_t*>(ngh_mask.data_ptr()) : nullptr,
                              node_degs.data_ptr<int32_t>(), length ? out_id.data_ptr<int32_t>() : nullptr,
                              length ? out_edge.data_ptr<int32_t>() : nullptr, static_cast<int>(id.numel()), length,
                              is_last ? 1 : 0, ws.data_ptr(), nbytes, nullptr, &valid_len, stream_of(id)),
          "mark_compact");
    auto info = torch::zeros({1}, torch::kFloat64);
    info[0] = static_cast<double>(valid_len);
    return {out_id, out_edge, info};
}

int get_map_back_part_size(Tensor node_deg, int valid_len)
{
    int fell_back = 0;
    const int ps = eppgcn_auto_back_part_size(valid_nodes(node_deg), valid_len, &fell_back);
    if (fell_back)
        TORCH_WARN_ONCE("get_map_back_part_size: the fitted regression gives a group size below 1 for this path (it "
                        "was fitted on small graphs); using the rule fitted for the wave64 kernels instead: ", ps);
    return ps;
}

// The group-size rule re-fitted for the wave64 kernels (no counterpart in the reference's module).
int get_wave64_back_part_size(Tensor node_deg, int valid_len)
{
    return eppgcn_wave64_back_part_size(valid_nodes(node_deg), valid_len);
}

std::vector<Tensor> split_back_part(Tensor node_deg, int num_edges, int back_part_size)
{
    auto s = split(node_deg, num_edges, back_part_size);
    auto info = torch::zeros({1}, torch::kInt32);
    info[0] = static_cast<int>(s.num_parts);
    return {s.part_pointer, info};
}

// Legacy all-in-one (EPPGCN.cpp:229-280): compaction, threshold rule when back_part_size == 0, split.
std::vector<Tensor> build_back_part(Tensor edge_mask, Tensor column_index, Tensor node_deg, int back_part_size, int dim)
{
    (void)dim;
    auto c = compact(edge_mask, column_index);
    if (back_part_size == 0) {
        back_part_size = eppgcn_threshold_back_part_size(valid_nodes(node_deg), c.valid_len);
        TORCH_CHECK(back_part_size > 0, "build_back_part: the threshold rule has no group size for an average kept "
                                        "degree >= 512; pass back_part_size explicitly");
    }
    auto s = split(node_deg, edge_mask.numel(), back_part_size);
    auto info = torch::zeros({2}, torch::kFloat64);
    info[0] = static_cast<double>(back_part_size);
    info[1] = static_cast<double>(s.num_parts);
    return {c.id, c.edge_list, s.part_pointer, info};
}

Tensor get_ginfo(Tensor node_deg, int valid_len)
{
    // the reference reads node_deg on the host (EPPGCN.cpp:351-386) and its caller passes a CPU tensor
    TORCH_CHECK(node_deg.scalar_type() == torch::kInt32, "node_deg must be int32");
    if (!node_deg.is_cuda()) node_deg = node_deg.to(torch::kCUDA);
    node_deg = node_deg.contiguous();
    CHECK_I32(node_deg);
    auto hist = torch::empty({10}, node_deg.options());
    auto re = torch::zeros({10}, torch::kFloat32);
    check(eppgcn_get_ginfo(i32(node_deg), node_deg.numel(), valid_len, hist.data_ptr<int32_t>(), re.data_ptr<float>(),
                           stream_of(node_deg)),
          "get_ginfo");
    return re;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    namespace py = pybind11;
    // the trailing keyword arguments are additions: relu_input applies max(x, 0) to the layer input
    // inside the product (and masks dX accordingly); need_dx=False skips dX (an empty tensor is returned)
    m.def("forward", &forward, "neighbour-group forward: X*W + aggregation (HIP)", py::arg("input"), py::arg("weight"),
          py::arg("row_pointers"), py::arg("column_index"), py::arg("degrees"), py::arg("part_pointers"),
          py::arg("part2Node"), py::arg("partSize"), py::arg("dimWorker"), py::arg("warpPerBlock"),
          py::arg("relu_input") = false);
    m.def("backward", &backward, "unpruned backward: aggregation + dX, dW (HIP)", py::arg("d_output"), py::arg("X"),
          py::arg("W"), py::arg("row_pointers"), py::arg("column_index"), py::arg("degrees"), py::arg("part_pointers"),
          py::arg("part2Node"), py::arg("partSize"), py::arg("dimWorker"), py::arg("warpPerBlock"),
          py::arg("need_dx") = true, py::arg("relu_input") = false);
    m.def("mask_forward", &mask_forward, "mark the backward execution path of one layer (HIP)");
    m.def("ours_backward", &ours_backward, "pruned backward over the compacted path: aggregation + dX, dW (HIP)",
          py::arg("d_output"), py::arg("X"), py::arg("W"), py::arg("id"), py::arg("partPointer"), py::arg("edgeList"),
          py::arg("degrees"), py::arg("partSize"), py::arg("numParts"), py::arg("layer"), py::arg("blockx"),
          py::arg("blocky"), py::arg("need_dx") = true, py::arg("relu_input") = false);
    m.def("set_dense_policy", [](int policy) { g_dense_policy = policy; },
          "dense products: 0 = library kernels where the shapes fit (default), -1 = always torch::mm");
    m.def("set_masked_update", [](bool on) { g_masked_update = on ? 1 : 0; },
          "pruned backward: true (default) = the dense products take the bitmap of the rows the aggregation wrote and the "
          "other rows are neither cleared nor read; false = clear and read every row");
    m.def("print_time", &eppgcn_print_time, "print accumulated kernel times");
    m.def("clear_time", &eppgcn_clear_time, "reset accumulated kernel times");
    m.def("set_timing", [](bool on) { eppgcn_set_timing(on ? 1 : 0); }, "enable per-call kernel timing");
    m.def("aggregation_status",
          []() { check(eppgcn_aggregation_status(static_cast<void*>(c10::hip::getCurrentHIPStream().stream())), "aggregation_status"); },
          "synchronise and raise if a planned aggregation call found its plan's memory replaced (see eppgcn_hip.h)");
    m.def("get_time_ms", &eppgcn_get_time_ms, "accumulated kernel time in ms");
    m.def("clear_plans", []() { drop_all_plans(); g_path_choices.clear(); }, "drop the cached execution plans");
    m.def("set_plan_policy", [](int policy) { g_plan_policy = policy; drop_all_plans(); g_path_choices.clear(); },
          "execution plans: 0 = where the feature table outgrows the caches (default), 1 = always, -1 = never");
    m.def("cached_plans", []() { return static_cast<int>(g_plans.size()); }, "number of execution plans held");
    m.def("cached_paths", []() { return static_cast<int>(g_path_choices.size()); }, "number of backward paths remembered");

    m.def("nll_forward", &nll_forward, "mean negative log-likelihood of the training rows (HIP)", py::arg("logits"),
          py::arg("rows"), py::arg("labels"));
    m.def("nll_backward", &nll_backward, "gradient of nll_forward (HIP)", py::arg("d_loss"), py::arg("logits"),
          py::arg("labels"), py::arg("num_rows"));
    m.def("gcn_layer", torch::wrap_pybind_function(gcn_layer), "forward of a layer with its autograd function in native code (HIP); None: not for these inputs",
          py::arg("input"), py::arg("weight"), py::arg("info"), py::arg("back"), py::arg("relu_input"));
    m.def("training_loss", torch::wrap_pybind_function(training_loss), "nll_forward with its autograd function in native code (HIP); None: not for these inputs",
          py::arg("logits"), py::arg("rows"), py::arg("labels"));
    GNNAFunctionBackward::add("GNNAFunctionBackward");
    TrainingLossBackward::add("_TrainingLossBackward");
    m.def("gradient_stays_unseen", &gradient_stays_unseen, "the loss is training_loss's own and has no hooks on its node");
    // what the two call, for callers that replace functions of this module
    m.attr("native_functions") = py::make_tuple(m.attr("forward"), m.attr("backward"), m.attr("ours_backward"),
                                                m.attr("nll_forward"), m.attr("nll_backward"));
    m.def("drop_gradients", &drop_gradients, "sets the gradients of the weights to None, as torch's zero_grad does");
    m.def("adam_step", &adam_step, "one Adam step of all weights in one launch (HIP); False: not this form, nothing changed");
    m.def("build_part", &build_part, "forward neighbour groups (HIP)");
    m.def("build_back_part", &build_back_part, "compaction + group split in one call (HIP)");
    m.def("compact_back_edge", &compact_back_edge, "compact the kept edges of one layer (HIP)");
    m.def("mark_compact", &mark_compact, "marking + compaction of one layer in one pass (HIP)");
    m.def("get_map_back_part_size", &get_map_back_part_size, "backward group size from the fitted regression");
    m.def("get_wave64_back_part_size", &get_wave64_back_part_size, "backward group size re-fitted for wave64 kernels");
    m.def("split_back_part", &split_back_part, "split kept edges into backward groups (HIP)");
    m.def("get_ginfo", &get_ginfo, "degree-distribution features of the kept path");
}

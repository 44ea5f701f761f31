// extern "C" entry points of libeppgcn_hip.so: argument checks, timers and the
// host halves (count read-back, heuristics) of the aggregation path.
#include "../../include/eppgcn_hip_tuning.h"

#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>

#include "common.hpp"

namespace eppgcn {

// ---- implemented in aggregate.hip / prepare.hip
int aggregate_forward_groups(float*, const float*, const int*, const float*, const int*, const int*, const void*, int,
                             int, int, int, float*, size_t, hipStream_t, double*, double*, bool out_is_clear = false);
int aggregate_compacted_groups(float*, const float*, const int*, const int*, const int*, const float*, const void*,
                               int, int, int, int, float*, size_t, const uint32_t*, hipStream_t, double*, double*,
                               const uint32_t** written = nullptr, long long* num_written = nullptr);
size_t plan_workspace_bytes(long long, long long);
int read_plan_status(const void*, long long, long long, long long, long long*, const void*, hipStream_t);
void set_stream_mode(int);
int last_call_used_stream();
int schedule_shift(int);
void set_schedule_shift(int);
void set_plan_keep_rows(int);
void set_plan_length_classes(int);
int check_plan_sizes(long long, long long, long long, size_t, size_t);
int launch_build_plan(const int*, const int*, const int*, const int*, int, long long, int, int, int, void*, size_t,
                      void*, size_t, const ScanState*, hipStream_t);
void set_agg_force_team(int);
void set_agg_force_rounds(int);
size_t feature_workspace_floats(long long, int);
int workspace_pitch(int);
int launch_dense_rows(float*, int, int, const float*, int, const float*, long long, long long, const float*,
                      const float*, int, int, long long, int, int, hipStream_t, unsigned, const uint32_t* rows = nullptr,
                      const RidingClear* clear = nullptr);
size_t update_workspace_bytes(long long, int, int);
int launch_dense_weight(float*, const float*, int, const float*, int, int, long long, int, int, void*, hipStream_t,
                        const uint32_t* rows = nullptr);
bool dense_backward_fused_covers(int, int, const float*, const float*);
int launch_dense_backward(float*, float*, const float*, const float*, const float*, int, long long, int, int, void*,
                          hipStream_t, const uint32_t* rows = nullptr);
size_t compact_workspace_bytes(long long);
size_t split_workspace_bytes(long long);
int launch_mask_forward(const int*, const int*, const int*, const uint8_t*, uint8_t*, int*, int*, int, long long, int,
                        hipStream_t);
int launch_compact_mask(const int*, int*, const int*, int*, long long, void*, hipStream_t);
long long static_compact_max_length();
int launch_compact_mask_static(const int*, int*, const int*, int*, long long, void**, hipStream_t);
int static_compact_workspace(void**);
int read_aggregation_status(hipStream_t);
size_t mark_compact_workspace_bytes(long long);
size_t mark_path_workspace_bytes(long long, long long);
size_t nll_workspace_bytes();
int launch_nll_forward(float*, const float*, const long long*, const int*, long long, long long, int, void*, hipStream_t);
int launch_nll_backward(float*, const float*, const float*, const int*, long long, long long, int, hipStream_t);
int launch_adam(int, float* const*, const float* const*, float* const*, float* const*, const long long*, const double*, double,
                double, double, double, hipStream_t);
uint8_t* mark_path_scratch(void*, long long, long long);
int launch_mark_path(const int*, const int*, const int*, const uint8_t*, uint8_t*, int*, int*, int*, uint32_t*, int,
                     long long, int, int, int, void*, hipStream_t);
int launch_mark_compact(const int*, const int*, const int*, const uint8_t*, uint8_t*, int*, int*, int*, int, long long,
                        int, void*, hipStream_t);
int launch_split(bool, const int*, int, int, int*, int*, long long, long long, bool, void*, hipStream_t);
int launch_gather_states(const void* const*, int, void*, hipStream_t);
int* plan_rows_in_workspace(void*, long long, long long);
const void* plan_header_address(const void*, long long, long long, long long);
int launch_count_nonzero(const int*, long long, int*, hipStream_t);
int launch_ginfo_hist(const int*, long long, int*, hipStream_t);
size_t mark_listed_rows_scratch_bytes(long long);
int launch_mark_listed_rows(const int*, long long, long long, uint32_t*, int*, uint8_t*, hipStream_t);
// ---- errors
static thread_local std::string g_last_error;
void set_error(const std::string& msg) { g_last_error = msg; }
int hip_fail(hipError_t e, const char* what)
{
    g_last_error = std::string(what) + ": " + hipGetErrorString(e);
    return kErrHip;
}

// ---- timers (milliseconds)
constexpr int kMaxTimedLayers = 16;
static std::atomic<bool> g_timing{false};
static double g_for_agg_ms = 0.0, g_back_agg_ms = 0.0, g_mask_ms = 0.0;
static double g_layer_back_ms[kMaxTimedLayers] = {0};

static double g_phase_ms[2] = {0.0, 0.0};       // output clears, pre-scaling passes of the aggregation calls

bool timing_enabled() { return g_timing.load(); }
double* phase_sink(int which) { return &g_phase_ms[which & 1]; }

// (read: a complete copy of the state that the caller already has on the host)
static int read_state(const void* workspace, hipStream_t stream, ScanState* host, const void* read = nullptr)
{
    if (read) {
        memcpy(host, read, sizeof(ScanState));
    } else {
        EPPGCN_HIP(hipMemcpyAsync(host, workspace, sizeof(ScanState), hipMemcpyDeviceToHost, stream));
        EPPGCN_HIP(hipStreamSynchronize(stream));
    }
    if (host->error) {
        set_error("look-back scan stalled: a tile waited past its spin limit; results are invalid");
        return kErrScanStalled;
    }
    return kOk;
}

// Bytes of a workspace whose head eppgcn_read_states copies: a whole record (kStateBytes), also where the call needs less (a
// split of up to 6144 vertices needs 40 to 56).  The calls that are older than the records still take what they need.
static size_t with_record(size_t bytes) { return bytes < kStateBytes ? kStateBytes : bytes; }

static bool aligned(const void* p, size_t a) { return reinterpret_cast<uintptr_t>(p) % a == 0; }

}  // namespace eppgcn

using namespace eppgcn;

extern "C" {

const char* eppgcn_last_error(void) { return g_last_error.c_str(); }
int eppgcn_abi_version(void) { return 20; }

// What the two unpruned aggregations refuse (`call` of them, or of a call that ends in one); reads nothing on the device.
static int check_spmm(const char* call, const float* out, const float* in, const int32_t* column_index, const float* degrees,
                      const int32_t* part_pointers, const int32_t* part2node, int num_nodes, int dim, int num_parts,
                      int part_size, int dim_worker, int warp_per_block, const float* workspace, size_t workspace_floats,
                      const void* plan)
{
    EPPGCN_REQUIRE_OF(call, num_nodes >= 0 && dim > 0 && num_parts >= 0, "num_nodes >= 0, dim > 0, num_parts >= 0 required");
    EPPGCN_REQUIRE_OF(call, part_size > 0 && dim_worker > 0 && warp_per_block > 0, "launch hints must be positive");
    if (num_nodes == 0) return kOk;
    EPPGCN_REQUIRE_OF(call, out && (in || workspace) && degrees, "null feature or scale pointer");
    EPPGCN_REQUIRE_OF(call, num_parts == 0 || (column_index && part_pointers && part2node), "null index pointer");
    EPPGCN_REQUIRE_OF(call, aligned(out, 4) && aligned(in, 4), "feature pointers must be 4-byte aligned");
    EPPGCN_REQUIRE_OF(call, !plan || aligned(plan, 256), "plan must be 256-byte aligned");
    EPPGCN_REQUIRE_OF(call, !workspace || (aligned(workspace, 16) && workspace != out),
                      "workspace must be 16-byte aligned and distinct from the output");
    EPPGCN_REQUIRE_OF(call, !workspace || workspace == in || workspace_floats >= feature_workspace_floats(num_nodes, dim),
                      "workspace smaller than eppgcn_feature_workspace_floats(num_nodes, dim)");
    return kOk;
}

int eppgcn_spmm_forward(float* out, const float* in, const int32_t* row_pointers, const int32_t* column_index,
                        const float* degrees, const int32_t* part_pointers, const int32_t* part2node, int num_nodes,
                        int dim, int num_parts, int part_size, int dim_worker, int warp_per_block, float* workspace,
                        size_t workspace_floats, const void* plan, void* stream)
{
    (void)row_pointers;
    if (int rc = check_spmm(__func__, out, in, column_index, degrees, part_pointers, part2node, num_nodes, dim, num_parts,
                            part_size, dim_worker, warp_per_block, workspace, workspace_floats, plan))
        return rc;
    if (num_nodes == 0) return kOk;
    return aggregate_forward_groups(out, in, column_index, degrees, part_pointers, part2node, plan, num_nodes, dim,
                                    num_parts, part_size, workspace, workspace_floats, static_cast<hipStream_t>(stream),
                                    &g_for_agg_ms, nullptr);
}

int eppgcn_spmm_backward(float* d_input, const float* d_output, const int32_t* row_pointers,
                         const int32_t* column_index, const float* degrees, const int32_t* part_pointers,
                         const int32_t* part2node, int num_nodes, int dim, int num_parts, int part_size, int dim_worker,
                         int warp_per_block, float* workspace, size_t workspace_floats, const void* plan, void* stream)
{
    (void)row_pointers;
    if (int rc = check_spmm(__func__, d_input, d_output, column_index, degrees, part_pointers, part2node, num_nodes, dim,
                            num_parts, part_size, dim_worker, warp_per_block, workspace, workspace_floats, plan))
        return rc;
    if (num_nodes == 0) return kOk;
    return aggregate_forward_groups(d_input, d_output, column_index, degrees, part_pointers, part2node, plan,
                                    num_nodes, dim, num_parts, part_size, workspace, workspace_floats,
                                    static_cast<hipStream_t>(stream), &g_back_agg_ms, nullptr);
}

// shared by the two pruned-backward entry points; written == nullptr: the plain call (every row of d_input defined)
static int ours_backward_call(float* d_input, const float* d_output, const int32_t* ids, const int32_t* part_pointer,
                              const int32_t* edge_list, const float* degrees, int num_nodes, int dim, int num_parts,
                              int part_size, int layer, int blockx, int blocky, float* workspace,
                              size_t workspace_floats, const void* plan, const uint32_t* gathered_rows,
                              const uint32_t** written, long long* num_written, void* stream)
{
    // part_size only sizes the work per wave (the reference's kernel ignores it, EPPGCN_kernel.cu:636)
    EPPGCN_REQUIRE(num_nodes >= 0 && dim > 0 && num_parts >= 0, "num_nodes >= 0, dim > 0, num_parts >= 0 required");
    EPPGCN_REQUIRE(blockx > 0 && blocky > 0, "launch hints must be positive");
    EPPGCN_REQUIRE(layer >= 1, "layer is 1-based");
    if (num_nodes == 0) return kOk;
    EPPGCN_REQUIRE(d_input && (d_output || workspace) && degrees, "null feature or scale pointer");
    EPPGCN_REQUIRE(num_parts == 0 || (ids && part_pointer && edge_list), "null index pointer");
    EPPGCN_REQUIRE(aligned(d_input, 4) && aligned(d_output, 4), "feature pointers must be 4-byte aligned");
    EPPGCN_REQUIRE(!plan || aligned(plan, 256), "plan must be 256-byte aligned");
    EPPGCN_REQUIRE(!workspace || (aligned(workspace, 16) && workspace != d_input),
                   "workspace must be 16-byte aligned and distinct from the output");
    EPPGCN_REQUIRE(!workspace || workspace == d_output || workspace_floats >= feature_workspace_floats(num_nodes, dim),
                   "workspace smaller than eppgcn_feature_workspace_floats(num_nodes, dim)");
    return aggregate_compacted_groups(d_input, d_output, ids, part_pointer, edge_list, degrees, plan, num_nodes,
                                      dim, num_parts, part_size > 0 ? part_size : 1, workspace, workspace_floats, gathered_rows,
                                      static_cast<hipStream_t>(stream), &g_back_agg_ms,
                                      layer <= kMaxTimedLayers ? &g_layer_back_ms[layer - 1] : nullptr, written, num_written);
}

int eppgcn_ours_backward(float* d_input, const float* d_output, const int32_t* ids, const int32_t* part_pointer,
                         const int32_t* edge_list, const float* degrees, int num_nodes, int dim, int num_parts,
                         int part_size, int layer, int blockx, int blocky, float* workspace,
                         size_t workspace_floats, const void* plan, const uint32_t* gathered_rows, void* stream)
{
    return ours_backward_call(d_input, d_output, ids, part_pointer, edge_list, degrees, num_nodes, dim, num_parts, part_size,
                              layer, blockx, blocky, workspace, workspace_floats, plan, gathered_rows, nullptr, nullptr, stream);
}

int eppgcn_ours_backward_rows(float* d_input, const float* d_output, const int32_t* ids, const int32_t* part_pointer,
                              const int32_t* edge_list, const float* degrees, int num_nodes, int dim, int num_parts,
                              int part_size, int layer, int blockx, int blocky, float* workspace,
                              size_t workspace_floats, const void* plan, const uint32_t* gathered_rows,
                              const uint32_t** written_rows, int64_t* num_written, void* stream)
{
    EPPGCN_REQUIRE(written_rows, "written_rows must not be NULL (eppgcn_ours_backward is the call without it)");
    *written_rows = nullptr;
    if (num_written) *num_written = num_nodes > 0 ? num_nodes : 0;
    long long count = num_nodes;
    const int rc = ours_backward_call(d_input, d_output, ids, part_pointer, edge_list, degrees, num_nodes, dim, num_parts,
                                      part_size, layer, blockx, blocky, workspace, workspace_floats, plan, gathered_rows,
                                      written_rows, &count, stream);
    if (rc == kOk && num_written && *written_rows) *num_written = count;
    return rc;
}

int eppgcn_mask_forward(const int32_t* part2node, const int32_t* part_pointers, const int32_t* column_index,
                        const uint8_t* src_mask, uint8_t* ngh_mask, int32_t* back_edge_mask, int32_t* node_degs,
                        int num_parts, int64_t num_edges, int is_last_layer, int blockx, int blocky, void* stream)
{
    EPPGCN_REQUIRE(num_parts >= 0 && num_edges >= 0, "negative size");
    EPPGCN_REQUIRE(blockx > 0 && blocky > 0, "launch hints must be positive");
    if (num_parts == 0) return kOk;
    EPPGCN_REQUIRE(part2node && part_pointers && column_index && src_mask && back_edge_mask && node_degs,
                   "null pointer");
    EPPGCN_REQUIRE(is_last_layer || ngh_mask, "ngh_mask may only be NULL on the last layer");
    KernelTimer t(static_cast<hipStream_t>(stream), &g_mask_ms);
    return launch_mask_forward(part2node, part_pointers, column_index, src_mask, ngh_mask, back_edge_mask, node_degs,
                               num_parts, num_edges, is_last_layer ? 1 : 0, static_cast<hipStream_t>(stream));
}

size_t eppgcn_feature_workspace_floats(int64_t num_nodes, int dim)
{
    return (num_nodes <= 0 || dim <= 0) ? 0 : feature_workspace_floats(num_nodes, dim);
}
int eppgcn_plan_recommended(int64_t num_nodes, int dim)
{
    if (num_nodes <= 0 || dim <= 0) return 0;
    return static_cast<double>(feature_workspace_floats(num_nodes, dim)) * 4.0 >= 4.0 * (1 << 20) ? 1 : 0;
}
size_t eppgcn_plan_bytes(int64_t num_parts, int64_t num_slots, int64_t num_nodes)
{
    return plan_bytes(num_parts, num_slots, num_nodes);
}
size_t eppgcn_plan_workspace_bytes(int64_t num_parts, int64_t num_slots)
{
    return plan_workspace_bytes(num_parts, num_slots);
}

static int check_plan_call(const char* call, const int32_t* part_pointers, const int32_t* column_index, const int32_t* part2node,
                           const int32_t* ids, int num_parts, int64_t num_slots, int num_nodes, int dim, int block_shift,
                           const void* plan, const void* workspace)
{
    EPPGCN_REQUIRE_OF(call, num_parts >= 0 && num_slots >= 0 && num_nodes >= 0 && dim > 0, "negative size");
    EPPGCN_REQUIRE_OF(call, block_shift >= 0 && block_shift <= 31, "block_shift must be 0 (automatic) or 1..31");
    if (num_parts == 0) return kOk;
    EPPGCN_REQUIRE_OF(call, part_pointers && column_index && plan, "null pointer");
    EPPGCN_REQUIRE_OF(call, (part2node != nullptr) != (ids != nullptr), "give exactly one of part2node (forward) and ids (backward)");
    EPPGCN_REQUIRE_OF(call, aligned(plan, 256) && workspace && aligned(workspace, 256), "plan and workspace must be 256-byte aligned");
    return kOk;
}

int eppgcn_build_plan(const int32_t* part_pointers, const int32_t* column_index, const int32_t* part2node,
                      const int32_t* ids, int num_parts, int64_t num_slots, int num_nodes, int dim, int block_shift,
                      void* plan, size_t plan_size, void* workspace, size_t workspace_bytes, void* stream)
{
    if (int rc = check_plan_call(__func__, part_pointers, column_index, part2node, ids, num_parts, num_slots, num_nodes, dim,
                                 block_shift, plan, workspace))
        return rc;
    if (num_parts == 0) return kOk;
    return launch_build_plan(part_pointers, column_index, part2node, ids, num_parts, num_slots, num_nodes,
                             block_shift > 0 ? block_shift : schedule_shift(dim), dim, plan, plan_size, workspace,
                             workspace_bytes, nullptr, static_cast<hipStream_t>(stream));
}

size_t eppgcn_compact_workspace_bytes(int64_t length) { return compact_workspace_bytes(length < 0 ? 0 : length); }
size_t eppgcn_split_workspace_bytes(int64_t num_nodes) { return with_record(split_workspace_bytes(num_nodes < 0 ? 0 : num_nodes)); }

int eppgcn_compact_back_edge(const int32_t* edge_mask, const int32_t* column_index, int32_t* out_id, int32_t* out_edge,
                             int64_t length, void* workspace, size_t workspace_bytes, int32_t* d_valid_len,
                             int64_t* h_valid_len, void* stream)
{
    EPPGCN_REQUIRE(length >= 0 && length < (1ll << 31), "length must fit int32");
    EPPGCN_REQUIRE(workspace && aligned(workspace, 8), "workspace must be 8-byte aligned");
    EPPGCN_REQUIRE(workspace_bytes >= compact_workspace_bytes(length), "workspace too small");
    EPPGCN_REQUIRE(length == 0 || (edge_mask && column_index && out_id && out_edge), "null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_compact_mask(edge_mask, out_id, column_index, out_edge, length, workspace, s)) return rc;
    ScanState* st = static_cast<ScanState*>(workspace);
    if (d_valid_len)
        EPPGCN_HIP(hipMemcpyAsync(d_valid_len, st->counts, sizeof(int), hipMemcpyDeviceToDevice, s));
    if (h_valid_len) {
        ScanState host;
        if (int rc = read_state(workspace, s, &host)) return rc;
        *h_valid_len = host.counts[0];
    }
    return kOk;
}

int64_t eppgcn_compact_back_edge_static_max_length(void) { return static_compact_max_length(); }

int eppgcn_compact_back_edge_static(const int32_t* edge_mask, const int32_t* column_index, int32_t* out_id,
                                    int32_t* out_edge, int64_t length, int32_t* d_valid_len, int64_t* h_valid_len,
                                    void* stream)
{
    EPPGCN_REQUIRE(length >= 0, "length must not be negative");
    if (length > static_compact_max_length()) {
        set_error("eppgcn_compact_back_edge_static: length " + std::to_string(length) + " exceeds the static scratch (" +
                  std::to_string(static_compact_max_length()) +
                  " slots at most); use eppgcn_compact_back_edge with a caller workspace");
        return kErrCapacity;
    }
    EPPGCN_REQUIRE(length == 0 || (edge_mask && column_index && out_id && out_edge), "null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    void* workspace = nullptr;
    if (int rc = launch_compact_mask_static(edge_mask, out_id, column_index, out_edge, length, &workspace, s)) return rc;
    ScanState* st = static_cast<ScanState*>(workspace);
    if (d_valid_len)
        EPPGCN_HIP(hipMemcpyAsync(d_valid_len, st->counts, sizeof(int), hipMemcpyDeviceToDevice, s));
    if (h_valid_len) {
        ScanState host;
        if (int rc = read_state(workspace, s, &host)) return rc;
        *h_valid_len = host.counts[0];
    }
    return kOk;
}

size_t eppgcn_mark_compact_workspace_bytes(int64_t num_edges) { return mark_compact_workspace_bytes(num_edges); }

int eppgcn_mark_compact(const int32_t* part2node, const int32_t* part_pointers, const int32_t* column_index,
                        const uint8_t* src_mask, uint8_t* ngh_mask, int32_t* node_degs, int32_t* out_id,
                        int32_t* out_edge, int num_parts, int64_t num_edges, int is_last, void* workspace,
                        size_t workspace_bytes, int32_t* d_valid_len, int64_t* h_valid_len, void* stream)
{
    EPPGCN_REQUIRE(num_parts >= 0 && num_edges >= 0 && num_edges < (1ll << 31), "num_parts >= 0 and 0 <= num_edges < 2^31 required");
    EPPGCN_REQUIRE(workspace && aligned(workspace, 8), "workspace must be 8-byte aligned");
    EPPGCN_REQUIRE(workspace_bytes >= mark_compact_workspace_bytes(num_edges), "workspace too small");
    EPPGCN_REQUIRE(num_edges == 0 || (out_id && out_edge), "null output pointer");
    EPPGCN_REQUIRE(num_parts == 0 || (part2node && part_pointers && column_index && src_mask && node_degs),
                   "null pointer");
    EPPGCN_REQUIRE(is_last || num_parts == 0 || ngh_mask, "ngh_mask is required unless this is the last layer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    {
        KernelTimer timer(s, &g_mask_ms);
        if (int rc = launch_mark_compact(part2node, part_pointers, column_index, src_mask, ngh_mask, node_degs, out_id,
                                         out_edge, num_parts, num_edges, is_last ? 1 : 0, workspace, s))
            return rc;
    }
    ScanState* st = static_cast<ScanState*>(workspace);
    if (d_valid_len)
        EPPGCN_HIP(hipMemcpyAsync(d_valid_len, st->counts, sizeof(int), hipMemcpyDeviceToDevice, s));
    if (h_valid_len) {
        ScanState host;
        if (int rc = read_state(workspace, s, &host)) return rc;
        *h_valid_len = host.counts[0];
    }
    return kOk;
}

size_t eppgcn_nll_workspace_bytes(void) { return nll_workspace_bytes(); }

int eppgcn_nll_forward(float* loss, const float* logits, const int64_t* rows, const int32_t* labels, int64_t num_rows,
                       int64_t num_nodes, int num_classes, void* workspace, size_t workspace_bytes, void* stream)
{
    EPPGCN_REQUIRE(num_rows >= 0 && num_nodes >= 0 && num_classes > 0, "negative size");
    EPPGCN_REQUIRE(num_rows == 0 || num_nodes > 0, "training rows of no vertices");
    EPPGCN_REQUIRE(loss && (num_rows == 0 || (logits && rows && labels)), "null pointer");
    EPPGCN_REQUIRE(workspace && aligned(workspace, 8) && workspace_bytes >= nll_workspace_bytes(), "workspace too small or not 8-byte aligned");
    static_assert(sizeof(long long) == sizeof(int64_t), "row ids are passed through");
    return launch_nll_forward(loss, logits, reinterpret_cast<const long long*>(rows), labels, num_rows, num_nodes, num_classes,
                              workspace, static_cast<hipStream_t>(stream));
}

int eppgcn_nll_backward(float* d_logits, const float* d_loss, const float* logits, const int32_t* labels, int64_t num_rows,
                        int64_t num_nodes, int num_classes, void* stream)
{
    EPPGCN_REQUIRE(num_rows >= 0 && num_nodes >= 0 && num_classes > 0, "negative size");
    EPPGCN_REQUIRE(num_nodes == 0 || (d_logits && d_loss && logits && labels), "null pointer");
    return launch_nll_backward(d_logits, d_loss, logits, labels, num_rows, num_nodes, num_classes,
                               static_cast<hipStream_t>(stream));
}

int eppgcn_adam_step(int count, float* const* params, const float* const* grads, float* const* exp_avg,
                     float* const* exp_avg_sq, const int64_t* sizes, const double* steps, double lr, double beta1,
                     double beta2, double eps, void* stream)
{
    EPPGCN_REQUIRE(count >= 0, "negative count");
    EPPGCN_REQUIRE(count == 0 || (params && grads && exp_avg && exp_avg_sq && sizes && steps), "null list");
    for (int k = 0; k < count; ++k) {
        EPPGCN_REQUIRE(sizes[k] >= 0 && steps[k] >= 1.0, "sizes must be >= 0 and steps >= 1");
        EPPGCN_REQUIRE(sizes[k] == 0 || (params[k] && grads[k] && exp_avg[k] && exp_avg_sq[k]), "null pointer");
        EPPGCN_REQUIRE(aligned(params[k], 4) && aligned(grads[k], 4) && aligned(exp_avg[k], 4) && aligned(exp_avg_sq[k], 4),
                       "pointers must be 4-byte aligned");
    }
    static_assert(sizeof(long long) == sizeof(int64_t), "sizes are passed through");
    return launch_adam(count, params, grads, exp_avg, exp_avg_sq, reinterpret_cast<const long long*>(sizes), steps, lr, beta1,
                       beta2, eps, static_cast<hipStream_t>(stream));
}

size_t eppgcn_mark_path_workspace_bytes(int64_t num_edges, int64_t num_nodes)
{
    return with_record(mark_path_workspace_bytes(num_edges < 0 ? 0 : num_edges, num_nodes < 0 ? 0 : num_nodes));
}

static int mark_path_call(const char* call, const int32_t* part2node, const int32_t* part_pointers, const int32_t* column_index,
                          const uint8_t* src_mask, uint8_t* ngh_mask, int32_t* node_degs, int32_t* out_id, int32_t* out_edge,
                          uint32_t* gathered_rows, int num_parts, int64_t num_edges, int num_nodes, int is_last, int part_size,
                          void* workspace, size_t workspace_bytes, void* stream)
{
    EPPGCN_REQUIRE_OF(call, num_parts >= 0 && num_nodes >= 0 && num_edges >= 0 && num_edges < (1ll << 31),
                      "num_parts, num_nodes >= 0 and 0 <= num_edges < 2^31 required");
    EPPGCN_REQUIRE_OF(call, part_size >= 0, "part_size >= 0 required");
    EPPGCN_REQUIRE_OF(call, workspace && aligned(workspace, 16), "workspace must be 16-byte aligned");
    EPPGCN_REQUIRE_OF(call, workspace_bytes >= mark_path_workspace_bytes(num_edges, num_nodes), "workspace too small");
    EPPGCN_REQUIRE_OF(call, num_edges == 0 || (out_id && out_edge), "null output pointer");
    EPPGCN_REQUIRE_OF(call, num_nodes == 0 || gathered_rows, "null output pointer");
    EPPGCN_REQUIRE_OF(call, num_parts == 0 || (part2node && part_pointers && column_index && src_mask && node_degs), "null pointer");
    EPPGCN_REQUIRE_OF(call, is_last || num_parts == 0 || ngh_mask, "ngh_mask is required unless this is the last layer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (num_parts == 0 || num_edges == 0 || num_nodes == 0) {
        if (num_nodes > 0)
            if (int rc = launch_zero_words(gathered_rows, (static_cast<size_t>(num_nodes) + 31) / 32, s)) return rc;
        if (num_edges > 0) {
            if (int rc = launch_zero_words(out_id, static_cast<size_t>(num_edges), s)) return rc;
            if (int rc = launch_zero_words(out_edge, static_cast<size_t>(num_edges), s)) return rc;
        }
        return launch_zero_words(workspace, sizeof(ScanState) / 4, s);
    }
    KernelTimer timer(s, &g_mask_ms);
    return launch_mark_path(part2node, part_pointers, column_index, src_mask, ngh_mask, node_degs, out_id, out_edge,
                            gathered_rows, num_parts, num_edges, num_nodes, is_last ? 1 : 0, part_size, workspace, s);
}

int eppgcn_mark_path(const int32_t* part2node, const int32_t* part_pointers, const int32_t* column_index,
                     const uint8_t* src_mask, uint8_t* ngh_mask, int32_t* node_degs, int32_t* out_id, int32_t* out_edge,
                     uint32_t* gathered_rows, int num_parts, int64_t num_edges, int num_nodes, int is_last, void* workspace,
                     size_t workspace_bytes, int64_t* counts, void* stream)
{
    if (int rc = mark_path_call(__func__, part2node, part_pointers, column_index, src_mask, ngh_mask, node_degs, out_id, out_edge,
                                gathered_rows, num_parts, num_edges, num_nodes, is_last, 0, workspace, workspace_bytes, stream))
        return rc;
    return counts ? eppgcn_mark_path_counts(out_edge, gathered_rows, num_edges, num_nodes, workspace, counts, stream) : kOk;
}

int eppgcn_mark_path_groups(const int32_t* part2node, const int32_t* part_pointers, const int32_t* column_index,
                            const uint8_t* src_mask, uint8_t* ngh_mask, int32_t* node_degs, int32_t* out_id,
                            int32_t* out_edge, uint32_t* gathered_rows, int num_parts, int64_t num_edges, int num_nodes,
                            int is_last, int part_size, void* workspace, size_t workspace_bytes, void* stream)
{
    EPPGCN_REQUIRE(workspace_bytes >= eppgcn_mark_path_workspace_bytes(num_edges, num_nodes), "workspace too small");
    return mark_path_call(__func__, part2node, part_pointers, column_index, src_mask, ngh_mask, node_degs, out_id, out_edge,
                          gathered_rows, num_parts, num_edges, num_nodes, is_last, part_size, workspace, workspace_bytes, stream);
}

int eppgcn_mark_path_counts(const int32_t* out_edge, uint32_t* gathered_rows, int64_t num_edges, int num_nodes,
                            void* workspace, int64_t* counts, void* stream)
{
    EPPGCN_REQUIRE(counts, "workspace (16-byte aligned) and counts required");
    int64_t four[4];
    counts[0] = counts[1] = counts[2] = 0;
    if (int rc = eppgcn_mark_path_group_counts(out_edge, gathered_rows, num_edges, num_nodes, workspace, nullptr, four, stream))
        return rc;
    for (int i = 0; i < 3; ++i) counts[i] = four[i];
    return kOk;
}

int eppgcn_mark_path_group_counts(const int32_t* out_edge, uint32_t* gathered_rows, int64_t num_edges, int num_nodes,
                                  void* workspace, const void* state, int64_t* counts, void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && num_edges >= 0 && num_edges < (1ll << 31), "num_nodes >= 0 and 0 <= num_edges < 2^31 required");
    EPPGCN_REQUIRE(workspace && aligned(workspace, 16) && counts, "workspace (16-byte aligned) and counts required");
    EPPGCN_REQUIRE((num_edges == 0 || out_edge) && (num_nodes == 0 || gathered_rows), "null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    counts[0] = counts[1] = counts[2] = counts[3] = 0;
    ScanState host;
    if (int rc = read_state(workspace, s, &host, state)) return rc;
    // the count sizes a launch below: a workspace that holds something else is told from it first
    if (host.counts[0] < 0 || host.counts[0] > num_edges || host.pad[2] < 0 || host.pad[2] > num_nodes || host.pad[0] < 0 ||
        host.pad[0] > num_nodes || host.counts[1] < 0 || host.counts[1] > host.counts[0]) {
        set_error("mark_path_counts: the workspace does not hold a finished eppgcn_mark_path of these sizes (it has to be called "
                  "with the same buffers and sizes, on the same stream)");
        return kErrInvalidArgument;
    }
    counts[0] = host.counts[0];
    counts[1] = host.pad[2];
    counts[2] = host.pad[0];
    counts[3] = host.counts[1];
    if (host.pad[1]) {          // a marked vertex without a kept self-loop: the gathered rows have to be looked for
        ScanState* st = static_cast<ScanState*>(workspace);
        if (int rc = launch_mark_listed_rows(out_edge, counts[0], num_nodes, gathered_rows, &st->pad[0],
                                             mark_path_scratch(workspace, num_edges, num_nodes), s))
            return rc;
        if (int rc = read_state(workspace, s, &host)) return rc;
        counts[2] = host.pad[0];
    }
    return kOk;
}

static int mark_gathered_call(const int32_t* edge_list, int64_t valid_len, int num_nodes, uint32_t* bitmap,
                              int32_t* d_count, int64_t* h_count, void* scratch, void* stream)
{
    EPPGCN_REQUIRE(valid_len >= 0 && valid_len < (1ll << 31) && num_nodes >= 0, "lengths must be non-negative int32");
    EPPGCN_REQUIRE(d_count && (num_nodes == 0 || bitmap) && (valid_len == 0 || edge_list), "null pointer");
    EPPGCN_REQUIRE(aligned(bitmap, 4) && aligned(d_count, 4), "bitmap and counter must be 4-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_mark_listed_rows(edge_list, valid_len, num_nodes, bitmap, d_count, static_cast<uint8_t*>(scratch), s))
        return rc;
    if (h_count) {
        int v = 0;
        EPPGCN_HIP(hipMemcpyAsync(&v, d_count, sizeof(int), hipMemcpyDeviceToHost, s));
        EPPGCN_HIP(hipStreamSynchronize(s));
        *h_count = v;
    }
    return kOk;
}

int eppgcn_mark_gathered_rows(const int32_t* edge_list, int64_t valid_len, int num_nodes, uint32_t* bitmap,
                              int32_t* d_count, int64_t* h_count, void* stream)
{
    return mark_gathered_call(edge_list, valid_len, num_nodes, bitmap, d_count, h_count, nullptr, stream);
}

size_t eppgcn_mark_gathered_rows_scratch_bytes(int64_t num_nodes)
{
    return num_nodes <= 0 ? 0 : mark_listed_rows_scratch_bytes(num_nodes);
}

int eppgcn_mark_gathered_rows_scratch(const int32_t* edge_list, int64_t valid_len, int num_nodes, uint32_t* bitmap,
                                      int32_t* d_count, int64_t* h_count, void* scratch, size_t scratch_bytes, void* stream)
{
    EPPGCN_REQUIRE(num_nodes <= 0 || (scratch && aligned(scratch, 16)), "scratch must be 16-byte aligned");
    EPPGCN_REQUIRE(num_nodes <= 0 || scratch_bytes >= mark_listed_rows_scratch_bytes(num_nodes), "scratch too small");
    return mark_gathered_call(edge_list, valid_len, num_nodes, bitmap, d_count, h_count, scratch, stream);
}

int eppgcn_count_nonzero(const int32_t* node_deg, int64_t length, int32_t* d_count, int64_t* h_count, void* stream)
{
    EPPGCN_REQUIRE(length >= 0 && length < (1ll << 31), "length must fit int32");
    EPPGCN_REQUIRE(d_count && (length == 0 || node_deg), "null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_count_nonzero(node_deg, length, d_count, s)) return rc;
    if (h_count) {
        int v = 0;
        EPPGCN_HIP(hipMemcpyAsync(&v, d_count, sizeof(int), hipMemcpyDeviceToHost, s));
        EPPGCN_HIP(hipStreamSynchronize(s));
        *h_count = v;
    }
    return kOk;
}

int eppgcn_map_back_part_size(int64_t valid_node, int64_t valid_len, int* clamped)
{
    if (clamped) *clamped = 0;
    if (valid_node <= 0) {
        if (clamped) *clamped = 1;
        return 1;
    }
    const double valid_degree = 1.0 * static_cast<double>(valid_len) / static_cast<double>(valid_node);
    const double beta0 = 0.65538, beta1 = 1.67431e-5, beta2 = -2.24342e-6, beta3 = 0.63641;
    const double raw = std::round(beta0 + beta1 * static_cast<double>(valid_node) +
                                  beta2 * static_cast<double>(valid_len) + beta3 * valid_degree);
    if (raw < 1.0) {
        if (clamped) *clamped = 1;
        return 1;
    }
    return static_cast<int>(raw);
}

int eppgcn_threshold_back_part_size(int64_t valid_node, int64_t valid_len)
{
    if (valid_node <= 0) return 4;
    const int64_t valid_degree = valid_len / valid_node;
    if (valid_degree < 4) return 4;
    if (valid_degree < 16) return 8;
    if (valid_degree < 64) return 16;
    if (valid_degree < 256) return 32;
    if (valid_degree < 512) return 64;
    return 0;
}

int eppgcn_wave64_back_part_size(int64_t valid_node, int64_t valid_len)
{
    // measured on R-MAT scale 20 and 22, mask ratios 0.01-0.5, widths 16-256: 16 is best or within 2 % of the
    // best up to an average kept degree of about 20, 32 above (first-layer paths with 30 kept edges per row:
    // 8 / 16 / 32 / 64 / 128 -> 1.97 / 1.42 / 1.21 / 1.30 / 1.63 ms)
    if (valid_node <= 0) return 16;
    return valid_len / valid_node < 24 ? 16 : 32;
}

int eppgcn_auto_back_part_size(int64_t valid_node, int64_t valid_len, int* fell_back)
{
    int clamped = 0;
    const int fitted = eppgcn_map_back_part_size(valid_node, valid_len, &clamped);
    if (fell_back) *fell_back = clamped;
    return clamped ? eppgcn_wave64_back_part_size(valid_node, valid_len) : fitted;
}

int eppgcn_scan_status(const void* workspace, void* stream)
{
    if (!workspace) {       // the static scratch of eppgcn_compact_back_edge_static on the current device
        void* ws = nullptr;
        if (int rc = static_compact_workspace(&ws)) return rc;
        workspace = ws;
    }
    EPPGCN_REQUIRE(aligned(workspace, 8), "workspace must be 8-byte aligned");
    ScanState host;
    if (int rc = read_state(const_cast<void*>(workspace), static_cast<hipStream_t>(stream), &host)) return rc;
    if (host.overflow) {
        set_error("group pointers did not fit the given capacity (need " + std::to_string(host.counts[0] + 1) +
                  " entries)");
        return kErrCapacity;
    }
    return kOk;
}

int eppgcn_plan_status(const void* plan, int num_parts, int64_t num_slots, int num_nodes, int64_t* partial_rows,
                       void* stream)
{
    EPPGCN_REQUIRE(num_parts >= 0 && num_slots >= 0 && num_nodes >= 0, "negative size");
    if (partial_rows) *partial_rows = 0;
    if (num_parts == 0) return kOk;
    EPPGCN_REQUIRE(plan && aligned(plan, 256), "plan must be 256-byte aligned");
    long long partial = 0;
    const int rc = read_plan_status(plan, num_parts, num_slots, num_nodes, &partial, nullptr, static_cast<hipStream_t>(stream));
    if (partial_rows) *partial_rows = partial;
    return rc;
}

const void* eppgcn_plan_state(const void* plan, int num_parts, int64_t num_slots, int num_nodes)
{
    return num_parts > 0 && num_slots >= 0 && num_nodes >= 0 && plan ? plan_header_address(plan, num_parts, num_slots, num_nodes)
                                                                     : nullptr;
}

int eppgcn_plan_status_read(const void* plan, int num_parts, int64_t num_slots, int num_nodes, const void* state,
                            int64_t* partial_rows)
{
    EPPGCN_REQUIRE(num_parts > 0 && num_slots >= 0 && num_nodes >= 0 && state, "num_parts > 0, sizes >= 0 and a state required");
    EPPGCN_REQUIRE(plan && aligned(plan, 256), "plan must be 256-byte aligned");
    long long partial = 0;
    const int rc = read_plan_status(plan, num_parts, num_slots, num_nodes, &partial, state, nullptr);
    if (partial_rows) *partial_rows = partial;
    return rc;
}

size_t eppgcn_state_bytes(void) { return kStateBytes; }

int eppgcn_read_states(const void* const* states, int count, void* host, void* stream)
{
    EPPGCN_REQUIRE(count >= 0 && (count == 0 || (states && host)), "null pointer");
    for (int i = 0; i < count; ++i) EPPGCN_REQUIRE(states[i] && aligned(states[i], 4), "every record must be a 4-byte aligned address");
    EPPGCN_REQUIRE(aligned(host, 4), "host memory must be 4-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_gather_states(states, count, host, s)) return rc;
    EPPGCN_HIP(hipStreamSynchronize(s));
    return kOk;
}

void eppgcn_plan_release(const void* plan)
{
    if (plan) forget_stream_info(plan);
}

int eppgcn_aggregation_status(void* stream) { return read_aggregation_status(static_cast<hipStream_t>(stream)); }

size_t eppgcn_plan_workspace_floats(const void* plan, int64_t num_nodes, int dim)
{
    size_t rows = static_cast<size_t>(swizzle_padded_rows(num_nodes));
    StreamInfo info;
    if (plan && find_stream_info(plan, &info) && info.header.valid) rows += static_cast<size_t>(info.header.num_partials);
    return rows * static_cast<size_t>(dim > 0 ? workspace_pitch(dim) : 0);
}

void eppgcn_set_stream_mode(int on) { set_stream_mode(on); }
int eppgcn_last_call_used_stream(void) { return last_call_used_stream(); }

static int finish_split(void* workspace, hipStream_t s, int32_t* d_counts, int64_t* h_a, int64_t* h_b, const void* read = nullptr)
{
    ScanState* st = static_cast<ScanState*>(workspace);
    if (d_counts) EPPGCN_HIP(hipMemcpyAsync(d_counts, st->counts, 2 * sizeof(int), hipMemcpyDeviceToDevice, s));
    if (h_a || h_b) {
        ScanState host;
        if (int rc = read_state(workspace, s, &host, read)) return rc;
        if (h_a) *h_a = host.counts[0];
        if (h_b) *h_b = host.counts[1];
        if (host.overflow) {
            set_error("group pointers do not fit the given capacity (need " + std::to_string(host.counts[0] + 1) +
                      " entries)");
            return kErrCapacity;
        }
    }
    return kOk;
}

int eppgcn_split_back_part(const int32_t* node_deg, int num_nodes, int part_size, int32_t* part_pointer,
                           int64_t capacity, void* workspace, size_t workspace_bytes, int32_t* d_counts,
                           int64_t* h_num_parts, int64_t* h_valid_len, void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && part_size >= 1, "num_nodes >= 0 and part_size >= 1 required");
    EPPGCN_REQUIRE(capacity >= 1 && part_pointer, "part_pointer needs at least one entry");
    EPPGCN_REQUIRE(workspace && aligned(workspace, 8), "workspace must be 8-byte aligned");
    EPPGCN_REQUIRE(workspace_bytes >= split_workspace_bytes(num_nodes), "workspace too small");
    EPPGCN_REQUIRE(num_nodes == 0 || node_deg, "null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_split(false, node_deg, num_nodes, part_size, part_pointer, nullptr, capacity, 0, true, workspace, s))
        return rc;
    return finish_split(workspace, s, d_counts, h_num_parts, h_valid_len);
}

int eppgcn_split_counts(const void* workspace, int64_t* h_num_parts, int64_t* h_valid_len, void* stream)
{
    EPPGCN_REQUIRE(workspace && aligned(workspace, 8), "workspace must be 8-byte aligned");
    return finish_split(const_cast<void*>(workspace), static_cast<hipStream_t>(stream), nullptr, h_num_parts, h_valid_len);
}

int eppgcn_split_counts_read(const void* state, int64_t* h_num_parts, int64_t* h_valid_len)
{
    EPPGCN_REQUIRE(state && h_num_parts && h_valid_len, "null pointer");
    return finish_split(nullptr, nullptr, nullptr, h_num_parts, h_valid_len, state);
}

int eppgcn_split_and_plan(const int32_t* node_deg, const int32_t* edge_list, int num_nodes, int part_size,
                          int32_t* part_pointer, int64_t capacity, int num_parts, int64_t num_slots, int dim, int block_shift,
                          void* plan, size_t plan_bytes, void* workspace, size_t workspace_bytes, void* split_workspace,
                          size_t split_workspace_bytes_, void* stream)
{
    EPPGCN_REQUIRE(num_nodes > 0 && part_size >= 1 && num_parts > 0 && dim > 0, "num_nodes, part_size, num_parts, dim > 0 required");
    EPPGCN_REQUIRE(capacity > num_parts && part_pointer && node_deg, "part_pointer needs num_parts + 1 entries");
    EPPGCN_REQUIRE(split_workspace && aligned(split_workspace, 8), "workspace must be 8-byte aligned");
    EPPGCN_REQUIRE(split_workspace_bytes_ >= eppgcn_split_workspace_bytes(num_nodes), "workspace too small");
    // everything that the plan's build refuses is refused before the split is launched; the build keeps the groups' rows in
    // its workspace, where the split leaves them
    int* rows = num_slots >= 0 ? plan_rows_in_workspace(workspace, num_parts, num_slots) : nullptr;
    if (int rc = check_plan_call(__func__, part_pointer, edge_list, rows, nullptr, num_parts, num_slots, num_nodes, dim,
                                 block_shift, plan, workspace))
        return rc;
    if (int rc = check_plan_sizes(num_parts, num_slots, num_nodes, plan_bytes, workspace_bytes)) return rc;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_split(false, node_deg, num_nodes, part_size, part_pointer, rows, capacity, num_parts, true,
                              split_workspace, s))
        return rc;
    return launch_build_plan(part_pointer, edge_list, rows, nullptr, num_parts, num_slots, num_nodes,
                             block_shift > 0 ? block_shift : schedule_shift(dim), dim, plan, plan_bytes, workspace,
                             workspace_bytes, static_cast<const ScanState*>(split_workspace), s);
}

int eppgcn_build_part(const int32_t* row_pointers, int num_nodes, int part_size, int32_t* part_pointers,
                      int32_t* part2node, int64_t capacity, void* workspace, size_t workspace_bytes, int32_t* d_counts,
                      int64_t* h_num_parts, void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && part_size >= 1, "num_nodes >= 0 and part_size >= 1 required");
    EPPGCN_REQUIRE(capacity >= 1 && part_pointers && (capacity == 1 || part2node), "output buffers required");
    EPPGCN_REQUIRE(workspace && aligned(workspace, 8), "workspace must be 8-byte aligned");
    EPPGCN_REQUIRE(workspace_bytes >= split_workspace_bytes(num_nodes), "workspace too small");
    EPPGCN_REQUIRE(row_pointers, "null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_split(true, row_pointers, num_nodes, part_size, part_pointers, part2node, capacity, capacity - 1,
                              false, workspace, s))
        return rc;
    return finish_split(workspace, s, d_counts, h_num_parts, nullptr);
}

int eppgcn_get_ginfo(const int32_t* node_deg, int64_t num_nodes, int64_t valid_len, int32_t* d_hist, float* h_out,
                     void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && num_nodes < (1ll << 31), "num_nodes must fit int32");
    EPPGCN_REQUIRE(d_hist && h_out && (num_nodes == 0 || node_deg), "null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_ginfo_hist(node_deg, num_nodes, d_hist, s)) return rc;
    int hist[10];
    EPPGCN_HIP(hipMemcpyAsync(hist, d_hist, sizeof(hist), hipMemcpyDeviceToHost, s));
    EPPGCN_HIP(hipStreamSynchronize(s));
    // same expressions as the reference: float counts, double divisions, float32 results
    const int valid_node = hist[0];
    h_out[0] = static_cast<float>(valid_node * 1.0 / 10000);
    h_out[1] = static_cast<float>(valid_len * 1.0 / 10000);
    h_out[2] = static_cast<float>(1.0 * valid_len / valid_node);
    for (int i = 3; i < 10; ++i) h_out[i] = static_cast<float>(static_cast<float>(hist[i]) * 1.0 / valid_node);
    return kOk;
}

void eppgcn_set_timing(int enabled) { g_timing.store(enabled != 0); }

void eppgcn_print_time(void)
{
    // same lines as the reference's print_time (EPPGCN_kernel.cu:96-106), in seconds
    std::printf("for_agg_time: %.6f\n", g_for_agg_ms / 1000);
    std::printf("back_agg_time: %.6f\n", g_back_agg_ms / 1000);
    for (int i = 0; i < kMaxTimedLayers && g_layer_back_ms[i] != 0.0; ++i)
        std::printf("l%d_back_agg_time: %.6f\n", i + 1, g_layer_back_ms[i] / 1000);
    std::printf("mask_time: %.6f\n", g_mask_ms / 1000);
    std::fflush(stdout);
}

void eppgcn_clear_time(void)
{
    // the marking time survives a clear, as in the reference (EPPGCN_kernel.cu:108-116): marking
    // runs once during warm-up and is still reported after the timed epochs
    g_for_agg_ms = 0.0;
    g_back_agg_ms = 0.0;
    for (double& v : g_layer_back_ms) v = 0.0;
    g_phase_ms[0] = g_phase_ms[1] = 0.0;
}

double eppgcn_get_time_ms(int which)
{
    if (which == 0) return g_for_agg_ms;
    if (which == 1) return g_back_agg_ms;
    if (which == 2) return g_mask_ms;
    if (which == 3 || which == 4) return g_phase_ms[which - 3];
    if (which > 100 && which <= 100 + kMaxTimedLayers) return g_layer_back_ms[which - 101];
    return -1.0;
}

void eppgcn_set_team_size(int lanes) { set_agg_force_team(lanes); }
void eppgcn_set_rounds(int rounds) { set_agg_force_rounds(rounds); }
void eppgcn_set_wide_index(int on) { set_force_wide_index(on != 0); }
void eppgcn_set_scan_test_mode(unsigned spin_limit, int mute_first_tile) { set_scan_test_mode(spin_limit, mute_first_tile); }
void eppgcn_set_plan_shift(int shift) { set_schedule_shift(shift); }
void eppgcn_set_plan_keep_rows(int groups) { set_plan_keep_rows(groups); }
void eppgcn_set_plan_length_classes(int on) { set_plan_length_classes(on); }

// ---- dense update
int eppgcn_feature_workspace_pitch(int dim) { return dim > 0 ? workspace_pitch(dim) : 0; }

int eppgcn_update_supported(int in_dim, int out_dim)
{
    if (in_dim <= 0 || out_dim <= 0) return 0;
    int mask = 0;
    if (in_dim <= 1024) mask |= 1;       // forward: reduction over in_dim
    if (out_dim <= 1024) mask |= 2;      // backward_input: reduction over out_dim
    if (out_dim <= 64) mask |= 4;        // backward_weight: gradient columns held in one block
    return mask;
}

int eppgcn_update_forward(float* out, int ld_out, const float* x, const float* w, const float* scale,
                          int relu_input, int64_t num_nodes, int in_dim, int out_dim, void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && in_dim > 0 && out_dim > 0, "num_nodes >= 0, in_dim > 0, out_dim > 0 required");
    EPPGCN_REQUIRE(ld_out >= out_dim, "ld_out must be at least out_dim");
    if (num_nodes == 0) return kOk;
    EPPGCN_REQUIRE(out && x && w, "null matrix pointer");
    EPPGCN_REQUIRE(aligned(out, 4) && aligned(x, 4) && aligned(w, 4), "matrix pointers must be 4-byte aligned");
    EPPGCN_REQUIRE(out != x, "the product cannot be written over its input");
    return launch_dense_rows(out, ld_out, ld_out, x, in_dim, w, out_dim, 1, scale, nullptr, 0, relu_input ? 1 : 0,
                             num_nodes, in_dim, out_dim, static_cast<hipStream_t>(stream), 0u);
}

static int check_forward_table(const char* call, const float* table, size_t table_floats, const float* x, const float* w,
                               const float* scale, int64_t num_nodes, int in_dim, int out_dim)
{
    EPPGCN_REQUIRE_OF(call, num_nodes >= 0 && in_dim > 0 && out_dim > 0, "num_nodes >= 0, in_dim > 0, out_dim > 0 required");
    if (num_nodes == 0) return kOk;
    EPPGCN_REQUIRE_OF(call, table && x && w && scale, "null pointer");
    EPPGCN_REQUIRE_OF(call, aligned(table, 16) && aligned(x, 4) && aligned(w, 4), "table must be 16-byte, matrices 4-byte aligned");
    EPPGCN_REQUIRE_OF(call, table != x, "the product cannot be written over its input");
    EPPGCN_REQUIRE_OF(call, num_nodes < (1ll << 31), "too many rows");
    EPPGCN_REQUIRE_OF(call, table_floats >= feature_workspace_floats(num_nodes, out_dim),
                      "table smaller than eppgcn_feature_workspace_floats(num_nodes, out_dim)");
    return kOk;
}

int eppgcn_update_forward_table(float* table, size_t table_floats, const float* x, const float* w, const float* scale,
                                int relu_input, int64_t num_nodes, int in_dim, int out_dim, void* stream)
{
    if (int rc = check_forward_table(__func__, table, table_floats, x, w, scale, num_nodes, in_dim, out_dim)) return rc;
    if (num_nodes == 0) return kOk;
    const int pitch = workspace_pitch(out_dim);
    return launch_dense_rows(table, pitch, pitch, x, in_dim, w, out_dim, 1, scale, nullptr, 0, relu_input ? 1 : 0,
                             num_nodes, in_dim, out_dim, static_cast<hipStream_t>(stream), kRowSwizzleMask);
}

static bool overlap(const float* a, size_t a_floats, const float* b, size_t b_floats)
{
    const uintptr_t p = reinterpret_cast<uintptr_t>(a), q = reinterpret_cast<uintptr_t>(b);
    return p < q + 4 * b_floats && q < p + 4 * a_floats;
}

int eppgcn_layer_forward(float* out, const float* x, const float* w, int relu_input, const int32_t* row_pointers,
                         const int32_t* column_index, const float* degrees, const int32_t* part_pointers,
                         const int32_t* part2node, int num_nodes, int in_dim, int out_dim, int num_parts, int part_size,
                         int dim_worker, int warp_per_block, float* workspace, size_t workspace_floats, const void* plan,
                         void* stream)
{
    (void)row_pointers;
    // everything that the product or the aggregation refuses is refused before the first launch
    if (int rc = check_forward_table(__func__, workspace, workspace_floats, x, w, degrees, num_nodes, in_dim, out_dim)) return rc;
    if (int rc = check_spmm(__func__, out, nullptr, column_index, degrees, part_pointers, part2node, num_nodes, out_dim,
                            num_parts, part_size, dim_worker, warp_per_block, workspace, workspace_floats, plan))
        return rc;
    if (num_nodes == 0) return kOk;
    const size_t n = static_cast<size_t>(num_nodes), words = n * out_dim;
    // an output that shares memory with an operand is cleared when the product has read it
    const bool rides = !plan && num_parts > 0 && words <= kRidingClearWords && !timing_enabled() &&
                       !overlap(out, words, x, n * in_dim) && !overlap(out, words, w, static_cast<size_t>(in_dim) * out_dim);
    const RidingClear clear = rides ? riding_clear(out, words) : RidingClear{};
    const int pitch = workspace_pitch(out_dim);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (int rc = launch_dense_rows(workspace, pitch, pitch, x, in_dim, w, out_dim, 1, degrees, nullptr, 0, relu_input ? 1 : 0,
                                   num_nodes, in_dim, out_dim, s, kRowSwizzleMask, nullptr, rides ? &clear : nullptr))
        return rc;
    return aggregate_forward_groups(out, nullptr, column_index, degrees, part_pointers, part2node, plan, num_nodes, out_dim,
                                    num_parts, part_size, workspace, workspace_floats, s, &g_for_agg_ms, nullptr, rides);
}

int64_t eppgcn_feature_workspace_row(int64_t vertex)
{
    return vertex < 0 ? -1 : static_cast<int64_t>((static_cast<uint64_t>(vertex) & ~0xffffffffull) |
                                                  swizzled_row(static_cast<unsigned>(vertex & 0xffffffffll)));
}

int eppgcn_update_backward_input(float* d_x, const float* g, const float* w, const float* relu_ref,
                                 int64_t num_nodes, int in_dim, int out_dim, void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && in_dim > 0 && out_dim > 0, "num_nodes >= 0, in_dim > 0, out_dim > 0 required");
    if (num_nodes == 0) return kOk;
    EPPGCN_REQUIRE(d_x && g && w, "null matrix pointer");
    EPPGCN_REQUIRE(aligned(d_x, 4) && aligned(g, 4) && aligned(w, 4) && aligned(relu_ref, 4),
                   "matrix pointers must be 4-byte aligned");
    EPPGCN_REQUIRE(d_x != g, "the product cannot be written over its input");
    // reduction over the out_dim columns of g; operand element (d, k) is w[k, d]
    return launch_dense_rows(d_x, in_dim, in_dim, g, out_dim, w, 1, out_dim, nullptr, relu_ref, in_dim, 0, num_nodes,
                             out_dim, in_dim, static_cast<hipStream_t>(stream), 0u);
}

size_t eppgcn_update_workspace_bytes(int64_t num_nodes, int in_dim, int out_dim)
{
    return update_workspace_bytes(num_nodes, in_dim, out_dim);
}

int eppgcn_update_backward_weight(float* d_w, const float* x, const float* g, int relu_input, int64_t num_nodes,
                                  int in_dim, int out_dim, void* workspace, size_t workspace_bytes, void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && in_dim > 0 && out_dim > 0, "num_nodes >= 0, in_dim > 0, out_dim > 0 required");
    EPPGCN_REQUIRE(d_w, "null output pointer");
    EPPGCN_REQUIRE(num_nodes == 0 || (x && g), "null matrix pointer");
    EPPGCN_REQUIRE(aligned(d_w, 4) && aligned(x, 4) && aligned(g, 4), "matrix pointers must be 4-byte aligned");
    EPPGCN_REQUIRE(num_nodes == 0 || (workspace && aligned(workspace, 4) &&
                                      workspace_bytes >= update_workspace_bytes(num_nodes, in_dim, out_dim)),
                   "workspace smaller than eppgcn_update_workspace_bytes(num_nodes, in_dim, out_dim)");
    return launch_dense_weight(d_w, x, in_dim, g, out_dim, relu_input ? 1 : 0, num_nodes, in_dim, out_dim, workspace,
                               static_cast<hipStream_t>(stream));
}

int eppgcn_update_backward(float* d_x, float* d_w, const float* x, const float* g, const float* w, int relu_input,
                           int64_t num_nodes, int in_dim, int out_dim, void* workspace, size_t workspace_bytes,
                           void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && in_dim > 0 && out_dim > 0, "num_nodes >= 0, in_dim > 0, out_dim > 0 required");
    EPPGCN_REQUIRE(d_w, "null output pointer");
    EPPGCN_REQUIRE(num_nodes == 0 || (d_x && x && g && w), "null matrix pointer");
    EPPGCN_REQUIRE(aligned(d_x, 4) && aligned(d_w, 4) && aligned(x, 4) && aligned(g, 4) && aligned(w, 4),
                   "matrix pointers must be 4-byte aligned");
    EPPGCN_REQUIRE(d_x != g && d_x != x, "the input gradient cannot be written over an input");
    EPPGCN_REQUIRE(num_nodes == 0 || (workspace && aligned(workspace, 4) &&
                                      workspace_bytes >= update_workspace_bytes(num_nodes, in_dim, out_dim)),
                   "workspace smaller than eppgcn_update_workspace_bytes(num_nodes, in_dim, out_dim)");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (num_nodes == 0 || dense_backward_fused_covers(in_dim, out_dim, x, g))
        return launch_dense_backward(d_x, d_w, x, g, w, relu_input ? 1 : 0, num_nodes, in_dim, out_dim, workspace, s);
    if (int rc = launch_dense_weight(d_w, x, in_dim, g, out_dim, relu_input ? 1 : 0, num_nodes, in_dim, out_dim,
                                     workspace, s))
        return rc;
    if (num_nodes == 0) return kOk;
    return launch_dense_rows(d_x, in_dim, in_dim, g, out_dim, w, 1, out_dim, nullptr, relu_input ? x : nullptr, in_dim,
                             0, num_nodes, out_dim, in_dim, s, 0u);
}

int eppgcn_update_backward_rows(float* d_x, float* d_w, const float* x, const float* g, const float* w, int relu_input,
                                const uint32_t* rows, int64_t num_nodes, int in_dim, int out_dim, void* workspace,
                                size_t workspace_bytes, void* stream)
{
    EPPGCN_REQUIRE(num_nodes >= 0 && in_dim > 0 && out_dim > 0, "num_nodes >= 0, in_dim > 0, out_dim > 0 required");
    EPPGCN_REQUIRE(d_w, "null output pointer");
    EPPGCN_REQUIRE(num_nodes == 0 || (x && g && (w || !d_x)), "null matrix pointer");
    EPPGCN_REQUIRE(aligned(d_x, 4) && aligned(d_w, 4) && aligned(x, 4) && aligned(g, 4) && aligned(w, 4) && aligned(rows, 4),
                   "matrix pointers and the row bitmap must be 4-byte aligned");
    EPPGCN_REQUIRE(!d_x || (d_x != g && d_x != x), "the input gradient cannot be written over an input");
    EPPGCN_REQUIRE(num_nodes == 0 || (workspace && aligned(workspace, 4) &&
                                      workspace_bytes >= update_workspace_bytes(num_nodes, in_dim, out_dim)),
                   "workspace smaller than eppgcn_update_workspace_bytes(num_nodes, in_dim, out_dim)");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (d_x && (num_nodes == 0 || dense_backward_fused_covers(in_dim, out_dim, x, g)))
        return launch_dense_backward(d_x, d_w, x, g, w, relu_input ? 1 : 0, num_nodes, in_dim, out_dim, workspace, s, rows);
    if (int rc = launch_dense_weight(d_w, x, in_dim, g, out_dim, relu_input ? 1 : 0, num_nodes, in_dim, out_dim,
                                     workspace, s, rows))
        return rc;
    if (num_nodes == 0 || !d_x) return kOk;
    return launch_dense_rows(d_x, in_dim, in_dim, g, out_dim, w, 1, out_dim, nullptr, relu_input ? x : nullptr, in_dim,
                             0, num_nodes, out_dim, in_dim, s, 0u, rows);
}

}  // extern "C"

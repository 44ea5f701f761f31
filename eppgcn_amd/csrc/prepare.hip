// Execution-path preparation for gfx950 (wave64): path marking from the train
// mask, single-pass stream compaction of the kept edges, splitting of the kept
// edges into backward neighbour groups, forward neighbour groups from the CSR
// row pointers, and the small counting kernels the group-size heuristics need.
//
// Replaces mask_forward_cuda_kernel (EPPGCN/GCNConv/EPPGCN_kernel.cu:351-388), the three
// live cuCompactor namespaces and the thrust scans (EPPGCN/GCNConv/cuCompactor.cu:42-48,
// :328-465, :467-621, :623-680) and the CPU loop of build_part
// (EPPGCN/GCNConv/EPPGCN.cpp:186-227).
//
// Both scans are single-pass "decoupled look-back" scans: a tile publishes its
// aggregate, then its wave 0 walks back over the predecessors' descriptors, 64
// per step, until it meets a tile whose inclusive prefix is known.  Lane ranks
// inside a wave come from a 64-bit ballot and mbcnt; no block-wide bit-sliced
// counting and no second pass over the input.
#include <atomic>
#include <mutex>

#include "common.hpp"

// Scan scratch of the allocation-free compaction entry point: one ScanState and one 64-bit tile
// descriptor per tile of compact_mask_kernel (16384 slots), for inputs of up to 2^30 slots (512 KiB + 32
// bytes per GPU, held until the process ends).  The name is a host-side stand-in; host code only ever uses
// the device address hipGetSymbolAddress returns for it (static_compact_scratch below).
constexpr long long kStaticCompactMaxLength = 1ll << 30;
constexpr long long kStaticCompactTile = 16384;
constexpr size_t kStaticCompactScratchBytes = 32 + 8 * static_cast<size_t>(kStaticCompactMaxLength / kStaticCompactTile);
static __device__ __align__(256) unsigned char scratch[kStaticCompactScratchBytes];

namespace eppgcn {

// ================================================================ scan state init
__global__ void scan_init_kernel(ScanState* st, uint64_t* desc, int num_tiles)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < num_tiles) desc[i] = kTileEmpty;
    if (i == 0) {
        st->counter = 0;
        st->error = 0;
        st->counts[0] = 0;
        st->counts[1] = 0;
        st->overflow = 0;
    }
}

// Test knob for the stall path: with tile 0 muted every look-back runs into its (then tiny) spin limit,
// raises the error flag and carries on, so the kernels still drain and the host sees EPPGCN_ERR_SCAN_STALLED.
static std::atomic<unsigned> g_scan_mode{0};     // process-wide test knob (tuning header)
unsigned scan_mode() { return g_scan_mode.load(); }
void set_scan_test_mode(unsigned spin_limit, int mute_first_tile)
{
    g_scan_mode.store((spin_limit & 0x7fffffffu) | (mute_first_tile ? 0x80000000u : 0u));
}

// ================================================================ shared pieces
// Counts end in one atomic per workgroup.  Device-scope atomics on one address serialise at about 12 ns
// each: with one per wave, a million vertices took 50 us of which 45 were the 4096 additions (now 5).
__device__ __forceinline__ void add_block_count(int local, int* __restrict__ d_count)
{
    __shared__ int s_part[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) local += __shfl_xor(local, off, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) s_part[threadIdx.x / kWave] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int sum = s_part[0] + s_part[1] + s_part[2] + s_part[3];
        if (sum) atomicAdd(d_count, sum);
    }
}

// bit j of the result: byte j of x is not zero
__device__ __forceinline__ unsigned nonzero_bytes(unsigned x)
{
    const unsigned top = (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u;
    return ((top >> 7) * 0x01020408u) >> 24 & 0xfu;
}

// Zeros from word `from` to word `end` by threads i0 < stride: 16-byte stores between the aligned ends.
__device__ __forceinline__ void zero_from(int* __restrict__ p, long long from, long long end, long long i0, long long stride)
{
    typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
    if (from >= end) return;
    const long long head = min(end - from, static_cast<long long>((16 - reinterpret_cast<uintptr_t>(p + from) % 16) % 16 / 4));
    const long long vecs = (end - from - head) / 4;
    uintx4* v = reinterpret_cast<uintx4*>(p + from + head);
    for (long long i = i0; i < vecs; i += stride) __builtin_nontemporal_store(uintx4{0u, 0u, 0u, 0u}, v + i);
    const long long tail = from + head + 4 * vecs;
    if (i0 < head) p[from + i0] = 0;
    if (i0 < end - tail) p[tail + i0] = 0;
}

// ================================================================ path marking
// A wave owns 64 consecutive forward groups (one per lane) and walks the contiguous slot range
// they cover 64 slots at a time, so that the column ids are read and the edge marks written
// with full-width coalesced accesses whatever the group lengths are.  The group (hence the
// row) of a slot is found by a 6-step search over the 64 group starts kept in LDS.  Kept
// slots are counted per group from the wave ballot, the counts of adjacent groups of one row
// are added across lanes, and one atomic per (wave, row) updates node_degs.
constexpr int kMaskBlock = 256;
constexpr int kMaskWaves = kMaskBlock / kWave;

__global__ __launch_bounds__(kMaskBlock) void mask_forward_kernel(
    const int* __restrict__ part2node, const int* __restrict__ part_ptr, const int* __restrict__ col,
    const uint8_t* __restrict__ src_mask, uint8_t* __restrict__ ngh_mask, int* __restrict__ back_edge_mask,
    int* __restrict__ node_degs, int num_parts, int is_last)
{
    __shared__ int s_beg[kMaskWaves][kWave + 1];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long g0 = (static_cast<long long>(blockIdx.x) * kMaskWaves + wave) * kWave;
    if (g0 >= num_parts) return;                       // wave-uniform; the LDS rows are wave-private
    const int ng = static_cast<int>(min(static_cast<long long>(kWave), num_parts - g0));

    int beg = 0, end = 0, row = -1;
    bool row_in_src = false;
    if (lane < ng) {
        beg = part_ptr[g0 + lane];
        end = part_ptr[g0 + lane + 1];
        row = part2node[g0 + lane];
        row_in_src = !is_last && end > beg && src_mask[row] != 0;
        if (row_in_src) ngh_mask[row] = 1;
    }
    int* begs = s_beg[wave];
    begs[lane] = lane < ng ? beg : 0x7fffffff;
    if (lane == 0) begs[kWave] = 0x7fffffff;
    __builtin_amdgcn_wave_barrier();
    const int first = __shfl(beg, 0, kWave);
    const int last = __shfl(end, ng - 1, kWave);

    int kept = 0;
    for (int base = first; base < last; base += kWave) {
        const int e = base + lane;
        const bool in_range = e < last;
        int owner = 0;
#pragma unroll
        for (int step = kWave / 2; step > 0; step >>= 1)
            if (begs[owner + step] <= e) owner += step;          // last group starting at or before e
        const int e_row = __shfl(row, owner, kWave);
        const bool e_src = __shfl(static_cast<int>(row_in_src), owner, kWave) != 0;
        bool keep = false;
        if (in_range) {
            const int end_id = col[e];
            keep = src_mask[end_id] != 0;
            if (keep) back_edge_mask[e] = e_row;
            if (e_src) ngh_mask[end_id] = 1;
        }
        const uint64_t ballot = __ballot(keep);
        // this lane's group covers wave slots [lo, hi) of the current 64
        const int lo = min(max(beg - base, 0), kWave);
        const int hi = min(max(end - base, 0), kWave);
        if (hi > lo) {
            const uint64_t below_hi = hi == kWave ? ~0ull : (1ull << hi) - 1ull;
            kept += __popcll(ballot & below_hi & ~((1ull << lo) - 1ull));
        }
    }
    // adjacent lanes whose groups belong to one row form a run: one atomic per run
    const int prev_row = __shfl_up(row, 1, kWave);
    const uint64_t heads = __ballot(lane == 0 || prev_row != row);
    kept = wave_run_sum(kept, heads);
    if (lane < ng && ((heads >> lane) & 1ull) && kept > 0) atomicAdd(node_degs + row, kept);
}

// ================================================================ compaction
constexpr int kCompactBlock = 256;
constexpr int kCompactItems = 16;
constexpr int kCompactTile = kCompactBlock * kCompactItems;
static_assert(kCompactItems * (kCompactBlock / kWave) == kWave, "one wave scans the per-(slab, wave) counts");

// Tile of the compaction kernel: kCompactMaskItems items per thread, 16384 per tile.  The tile-id counter is one line
// that every workgroup hits with a device-scope atomic, and those serialise; at R-MAT scale 22 (132 M slots) tiles of
// 4096 slots took 0.47 / 0.62 ms (a tenth / nearly all of the slots kept), tiles of 16384 take 0.38 / 0.53 ms.
// 16-byte loads of the mask with the same tile: 0.34 / 0.60 ms (each lane then stores 4 items of its own and a store
// instruction covers every fourth word) - not kept.
constexpr int kCompactMaskItems = 64;
constexpr int kCompactMaskTile = kCompactBlock * kCompactMaskItems;
static_assert(kCompactMaskTile % kCompactTile == 0, "the workspace is sized for tiles of kCompactTile slots");

__global__ __launch_bounds__(kCompactBlock) void compact_mask_kernel(
    const int* __restrict__ in_id, const int* __restrict__ in_edge, int* __restrict__ out_id,
    int* __restrict__ out_edge, int length, int num_tiles, ScanState* st, uint64_t* desc, unsigned mode)
{
    constexpr int kItems = kCompactMaskItems;
    constexpr int kWaves = kCompactBlock / kWave;
    constexpr int kPerLane = kItems * kWaves / kWave;        // counts a lane of the scanning wave adds up
    __shared__ int s_tile;
    __shared__ int s_count[kItems * kWaves];                 // (item k, wave) in output order
    __shared__ int s_prefix;
    const int tile = acquire_tile(st, &s_tile);
    if (tile >= num_tiles) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long base = static_cast<long long>(tile) * kCompactMaskTile;

    int v[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const long long idx = base + k * kCompactBlock + threadIdx.x;
        v[k] = idx < length ? in_id[idx] : -1;
    }
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const uint64_t ballot = __ballot(v[k] != -1);
        if (lane == 0) s_count[k * kWaves + wave] = __popcll(ballot);
    }
    __syncthreads();
    if (wave == 0) {
        int c[kPerLane], sum = 0;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            c[j] = s_count[lane * kPerLane + j];
            sum += c[j];
        }
        const int incl = wave_inclusive_scan(sum);
        const int total = __shfl(incl, kWave - 1, kWave);
        int run = incl - sum;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            s_count[lane * kPerLane + j] = run;
            run += c[j];
        }
        const uint64_t excl = tile_lookback(desc, st, tile, static_cast<uint64_t>(total), mode);
        if (lane == 0) {
            s_prefix = static_cast<int>(excl);
            if (tile == num_tiles - 1) st->counts[0] = static_cast<int>(excl) + total;
        }
    }
    __syncthreads();
    const int prefix = s_prefix;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const bool pred = v[k] != -1;
        const uint64_t ballot = __ballot(pred);
        if (pred) {
            const long long idx = base + k * kCompactBlock + threadIdx.x;
            const int dst = prefix + s_count[k * kWaves + wave] + ballot_rank(ballot);
            out_id[dst] = v[k];
            out_edge[dst] = in_edge[idx];
        }
    }
}

// ================================================================ marking + compaction in one pass
// What mask_forward_kernel followed by compact_mask_kernel do, without the E-entry edge mask between them, in two kernels
// over tiles of kMarkTile consecutive slots.
//   keep_slots_kernel    keep = the slot's column is in the source mask: one bit per slot and a count per tile.  Nothing but
//                        column ids and mask entries is read.  The lookups are what it takes (64 lines an instruction), and
//                        they run best with few of them under way per thread: 16, 8, 4 of each 312, 265, 254 us for 132 M slots.
//   scan_counts_kernel   (kMarkScannedTiles tiles and more) the kept slots before every tile, by one workgroup: 5.7 us for 32
//                        thousand tiles.  A workgroup per tile that adds up the counts before its own reads 2 tiles^2 bytes:
//                        0.13 GB, from L2, at the line, where either way takes the same time (7 thousand tiles 142 / 139 us
//                        with and without the scan, 16 thousand 374 / 353; 4 thousand 112 / 113, 900 36 / 39).
//   place_slots_kernel   rows and places of the kept slots; the row of a slot comes from a bit map of the group starts inside
//                        the tile (prefix population count; the tile's first group was found beforehand) and the rows of
//                        the tile's groups, staged in LDS; kept slots per row are differences of the prefix counts, one
//                        atomic per (wave, row): a hub of 600 thousand slots costs 150 tiles a few atomics each, where one
//                        per 64 slots queued ten thousand on one address.
constexpr int kMarkTile = 4096;           // slots of a tile
constexpr int kKeepBlock = 1024;
// Groups of a tile whose rows are staged (more, which takes empty groups: read where they are needed).  The first group of the next
// tile counts, so a tile of one-slot groups has one more than slots.  Without room for it, us for a whole marking: 34 M rows of
// one slot 832, now 503; R-MAT scale 22 in groups of one slot 2724, now 1530.
constexpr int kMarkStagedRows = kMarkTile + 1;
constexpr int kMarkScannedTiles = 8192;   // tiles from which on their counts are scanned by a launch of its own

typedef int int4u __attribute__((ext_vector_type(4), aligned(4)));

// first[t] = last group starting at or before slot t * kMarkTile (group 0 for slots before all groups); first[num_tiles] = last
// group.  Every group says so for the tiles whose first slot it holds: the pointers are read once, in order (a search per tile is
// a chain of 20 loads).  A thread takes four groups at a time; the tiles of a group that holds many, or of the last one when slots
// of no group follow it, are written by its wave (a whole marking of 2^27 slots in one group 1.70 -> 0.89 ms; one thread took
// 0.8 ms for the 32 thousand tiles).  All lanes of the wave have to be active.
__device__ __forceinline__ void mark_tile_groups(const int* __restrict__ part_ptr, int num_parts, int num_tiles,
                                                 int* __restrict__ first, int thread, int threads)
{
    constexpr int kGroups = 4;
    constexpr int kAlone = 4;                                // tiles that a thread writes itself
    const int lane = lane_id();
    for (long long w0 = static_cast<long long>(thread - lane) * kGroups; w0 < num_parts; w0 += static_cast<long long>(threads) * kGroups) {
        const long long g0 = w0 + lane * kGroups;
        int start[kGroups + 1];
#pragma unroll
        for (int j = 0; j <= kGroups; ++j) start[j] = part_ptr[min(g0 + j, static_cast<long long>(num_parts))];
#pragma unroll
        for (int j = 0; j < kGroups; ++j) {
            const long long g = g0 + j;
            const bool last = g == num_parts - 1;
            const int t0 = g == 0 ? 0 : static_cast<int>((static_cast<unsigned>(max(start[j], 0)) + (kMarkTile - 1u)) / kMarkTile);
            int t1 = min(num_tiles, static_cast<int>((static_cast<unsigned>(max(start[j + 1], 0)) + (kMarkTile - 1u)) / kMarkTile));
            if (last) t1 = num_tiles;
            if (g >= num_parts) t1 = 0;
            for (int t = t0; t < min(t1, t0 + kAlone); ++t) first[t] = static_cast<int>(g);
            if (last) first[num_tiles] = static_cast<int>(g);
            for (uint64_t more = __ballot(t1 - t0 > kAlone); more; more &= more - 1) {
                const int k = __builtin_ctzll(more);
                const int from = __builtin_amdgcn_readlane(t0, k) + kAlone, to = __builtin_amdgcn_readlane(t1, k);
                const int group = static_cast<int>(w0 + k * kGroups + j);
                for (int t = from + 4 * lane; t < to; t += 4 * kWave) {
                    if (t + 4 <= to) *reinterpret_cast<int4u*>(first + t) = int4u{group, group, group, group};
                    else
                        for (int i = t; i < to; ++i) first[i] = group;
                }
            }
        }
    }
}

__global__ __launch_bounds__(256) void tile_groups_kernel(const int* __restrict__ part_ptr, int num_parts, int num_tiles,
                                                          int* __restrict__ first, ScanState* st)
{
    const int i0 = blockIdx.x * 256 + threadIdx.x, stride = gridDim.x * 256;
    if (i0 == 0) *st = ScanState{};
    mark_tile_groups(part_ptr, num_parts, num_tiles, first, i0, stride);
}

// kBits: the source mask is read as bits (packed once per call): eight times as many vertices share a cache line
template <bool kBits>
__device__ __forceinline__ bool in_mask(const void* __restrict__ mask, int v)
{
    if constexpr (kBits) return ((static_cast<const uint32_t*>(mask)[static_cast<unsigned>(v) >> 5] >> (v & 31)) & 1u) != 0u;
    else return static_cast<const uint8_t*>(mask)[v] != 0;
}

template <bool kBits>
__global__ __launch_bounds__(kKeepBlock) void keep_slots_kernel(const int* __restrict__ part_ptr, const int* __restrict__ col,
                                                                const void* __restrict__ src, int num_parts, int length,
                                                                unsigned long long* __restrict__ kept, int* __restrict__ counts)
{
    constexpr int kItems = kMarkTile / kKeepBlock;
    constexpr int kWaves = kKeepBlock / kWave;
    constexpr int kWords = kMarkTile / 64;
    __shared__ unsigned long long s_kept[kWords];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long base = static_cast<long long>(blockIdx.x) * kMarkTile;
    // slots outside [part_ptr[0], part_ptr[num_parts]) belong to no group and are never kept
    const int owned_lo = part_ptr[0];
    const int owned_hi = min(part_ptr[num_parts], length);
    int c[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const long long idx = base + k * kKeepBlock + threadIdx.x;
        c[k] = idx >= owned_lo && idx < owned_hi ? col[idx] : -1;
    }
    bool keep[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k) keep[k] = in_mask<kBits>(src, max(c[k], 0));
    uint64_t mine = 0;                                       // lane k: the ballot of slot k
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const uint64_t ballot = __ballot(keep[k] && c[k] >= 0);
        if (lane == k) mine = ballot;
    }
    if (lane < kItems) s_kept[lane * kWaves + wave] = mine;
    __syncthreads();
    static_assert(kWords == kWave, "one wave takes the words of a tile");
    if (wave == 0) {
        const unsigned long long word = s_kept[lane];
        kept[static_cast<long long>(blockIdx.x) * kWords + lane] = word;
        const int n = wave_inclusive_scan(__popcll(word));
        if (lane == kWave - 1) counts[blockIdx.x] = n;
    }
}

// counts[0 .. n) become their exclusive prefix sums
__global__ __launch_bounds__(1024) void scan_counts_kernel(int* __restrict__ counts, int n)
{
    constexpr int kVecs = 4, kWaves = 1024 / kWave;          // vector (v, thread) of a step: 4 counts at (v * 1024 + thread) * 4
    __shared__ int s_wave[kVecs * kWaves];
    static_assert(kVecs * kWaves == kWave, "one wave scans the (vector, wave) sums");
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    int carry = 0;
    for (int t0 = 0; t0 < n; t0 += 4096 * kVecs) {
        int4u c[kVecs];
        int before[kVecs];
#pragma unroll
        for (int v = 0; v < kVecs; ++v) {
            const int t = t0 + (v * 1024 + static_cast<int>(threadIdx.x)) * 4;
            c[v] = int4u{0, 0, 0, 0};
            if (t + 4 <= n) c[v] = *reinterpret_cast<const int4u*>(counts + t);
            else
                for (int j = 0; j < 4; ++j) c[v][j] = t + j < n ? counts[t + j] : 0;
        }
#pragma unroll
        for (int v = 0; v < kVecs; ++v) {
            const int sum = c[v][0] + c[v][1] + c[v][2] + c[v][3];
            const int incl = wave_inclusive_scan(sum);
            before[v] = incl - sum;
            if (lane == kWave - 1) s_wave[v * kWaves + wave] = incl;
        }
        __syncthreads();
        const int mine = s_wave[lane], incl = wave_inclusive_scan(mine);
        const int excl = carry + incl - mine;                // lane v * kWaves + w: before wave w's vector v
#pragma unroll
        for (int v = 0; v < kVecs; ++v) {
            const int t = t0 + (v * 1024 + static_cast<int>(threadIdx.x)) * 4;
            int4u out;
            out[0] = __shfl(excl, v * kWaves + wave, kWave) + before[v];
            out[1] = out[0] + c[v][0];
            out[2] = out[1] + c[v][1];
            out[3] = out[2] + c[v][2];
            if (t + 4 <= n) *reinterpret_cast<int4u*>(counts + t) = out;
            else
                for (int j = 0; j < 4; ++j)
                    if (t + j < n) counts[t + j] = out[j];
        }
        carry += __builtin_amdgcn_readlane(incl, kWave - 1);
        __syncthreads();
    }
}

// Vector loads and stores of a wave are counted together and in order: a wait for a load waits for every store before it.  So a
// workgroup loads first - the columns of all its slots, then the groups - and stores last: neighbour marks, kept slots, counts
// per row, zeros.  A wave has consecutive slots, so that its stores share lines with its own next ones.  Slot by slot, each
// waiting for the stores of the one before it (and all of them for the zeros), in tiles of 16 384 slots, a layer of R-MAT scale
// 22 took 519 / 372 us (a tenth / 95 % of 132 M slots kept); now 454 / 331.  2253 tiles 52 / 44 -> 43 / 38, 27 tiles
// 13.5 -> 12.
template <int kBlock, bool kScanned, bool kBits>
__global__ __launch_bounds__(kBlock, 8) void place_slots_kernel(
    const int* __restrict__ part2node, const int* __restrict__ part_ptr, const int* __restrict__ col,
    const void* __restrict__ src, uint8_t* __restrict__ ngh_mask, int* __restrict__ node_degs, int* __restrict__ out_id,
    int* __restrict__ out_edge, uint8_t* __restrict__ self_kept, int num_parts, int length, int num_tiles, int is_last,
    const int* __restrict__ tile_first, const unsigned long long* __restrict__ kept, const int* __restrict__ counts,
    ScanState* st)
{
    constexpr int kTile = kMarkTile, kItems = kTile / kBlock;
    constexpr int kWords = kTile / 64;
    constexpr int kPerLane = kWords / kWave;
    constexpr int kBatch = kItems > 8 ? 1 : 2;           // groups a thread looks at together
    static_assert(kWords % kWave == 0 && kItems <= kWave, "one wave scans the words; a wave's words fit its lanes");
    static_assert(kWords <= kBlock && kBlock >= 2 * kWave, "a thread per word, a wave for each of the two maps");
    __shared__ int s_prefix;
    __shared__ int s_starts_in_tile;
    __shared__ unsigned long long s_starts[kWords];    // bit p: a group starts at slot base + p
    __shared__ unsigned long long s_kept[kWords];      // bit p: slot base + p is kept
    __shared__ int s_starts_before[kWords];            // group starts before each word
    __shared__ int s_kept_before[kWords + 1];          // kept slots before each word; [kWords] = all of the tile
    __shared__ unsigned s_row[kMarkStagedRows];        // rows of the tile's groups; bit 31: the row is in the source mask
    const int tile = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long base = static_cast<long long>(tile) * kTile;       // < length
    const int inside = static_cast<int>(min(static_cast<long long>(kTile), length - base));
    const int mine = wave * (kItems * kWave) + lane;      // this thread's first slot of the tile; the others are 64 apart
    int c[kItems];
    {
        const int* __restrict__ tile_col = col + base;
#pragma unroll
        for (int k = 0; k < kItems; ++k) c[k] = tile_col[min(mine + k * kWave, inside - 1)];
    }
    // in range for any pointers: a table of tiles whose groups do not ascend is left incomplete
    const int g_lo = min(max(tile_first[tile], 0), num_parts - 1);
    const int g_cnt = min(max(tile_first[tile + 1], g_lo), num_parts - 1) - g_lo + 1;
    const bool staged = g_cnt <= kMarkStagedRows;
    const int before = part_ptr[g_lo] < base ? 1 : 0;    // g_lo itself starts before the tile
    // slots of the tile that belong to groups: [owned_first, owned_first + owned_slots)
    const int owned_first = static_cast<int>(min(max(part_ptr[0] - base, 0ll), static_cast<long long>(kTile)));
    const unsigned owned_slots = static_cast<unsigned>(max(min(static_cast<int>(part_ptr[g_lo + g_cnt] - base), inside) - owned_first, 0));
    if (threadIdx.x < kWords) {
        s_starts[threadIdx.x] = 0ull;
        s_kept[threadIdx.x] = kept[static_cast<long long>(tile) * kWords + threadIdx.x];
    }
    if (threadIdx.x == 0) {
        s_starts_in_tile = 0;
        s_prefix = kScanned ? counts[tile] : 0;
    }
    __syncthreads();
    if constexpr (!kScanned) {
        int sum = 0;
        for (int t0 = threadIdx.x; t0 < tile; t0 += 4 * kBlock) {
            int n[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) n[j] = t0 + j * kBlock < tile ? counts[t0 + j * kBlock] : 0;
            sum += n[0] + n[1] + n[2] + n[3];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kWave);
        if (lane == 0 && sum) atomicAdd(&s_prefix, sum);
    }
    // the tile's groups, kBatch of them per thread at a time; the first of them (usually all) stay in registers
    struct Groups { int from[kBatch], to[kBatch]; };
    auto load_groups = [&](Groups& g, int i0) {
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int at = g_lo + min(i0 + j * kBlock + static_cast<int>(threadIdx.x), g_cnt - 1);
            g.from[j] = part_ptr[at];
            g.to[j] = part_ptr[at + 1];
        }
    };
    auto load_rows = [&](unsigned (&row)[kBatch], int i0) {        // bit 31: the row is in the source mask (never on the last layer)
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            row[j] = static_cast<unsigned>(part2node[g_lo + min(i0 + j * kBlock + static_cast<int>(threadIdx.x), g_cnt - 1)]);
        if (is_last) return;
        bool marked[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) marked[j] = in_mask<kBits>(src, static_cast<int>(row[j]));
#pragma unroll
        for (int j = 0; j < kBatch; ++j) row[j] |= marked[j] ? 0x80000000u : 0u;
    };
    Groups first;
    {
        int starts = 0;
        auto stage = [&](Groups& g, int i0) {
            unsigned row[kBatch];
            load_groups(g, i0);
            if (staged) load_rows(row, i0);
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int i = i0 + j * kBlock + static_cast<int>(threadIdx.x);
                if (i >= g_cnt) continue;
                const long long p = g.from[j] - base;
                if (p >= 0 && p < kTile) {
                    atomicOr(&s_starts[p >> 6], 1ull << (p & 63));
                    ++starts;
                }
                if (staged) s_row[i] = row[j];
            }
        };
        stage(first, 0);
        for (int i0 = kBlock * kBatch; i0 < g_cnt; i0 += kBlock * kBatch) {
            Groups g;
            stage(g, i0);
        }
        if (starts) atomicAdd(&s_starts_in_tile, starts);
    }
    __syncthreads();
    // The owner of slot e is g_lo - 1 + (number of groups of the tile that start at or before e).
    // When no two groups of the tile start at the same slot (no empty groups, as build_part guarantees) that number is a prefix
    // population count over the map of group starts; otherwise every slot does a binary search over the group starts.
    if (wave < 2) {
        const unsigned long long* words = wave == 0 ? s_kept : s_starts;
        int* out = wave == 0 ? s_kept_before : s_starts_before;
        int n[kPerLane], sum = 0;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            n[j] = __popcll(words[lane * kPerLane + j]);
            sum += n[j];
        }
        const int incl = wave_inclusive_scan(sum);
        int run = incl - sum;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            out[lane * kPerLane + j] = run;
            run += n[j];
        }
        if (lane == kWave - 1) {
            if (wave == 0) {
                s_kept_before[kWords] = incl;
                if (tile == num_tiles - 1) st->counts[0] = s_prefix + incl;
            } else if (incl != s_starts_in_tile) {
                s_starts_in_tile = -1;                       // duplicate starts
            }
        }
    }
    __syncthreads();
    // ---- the row of every slot
    const bool by_bits = s_starts_in_tile >= 0;
    // lane k: word k of this wave
    const int my_word = wave * kItems + (lane < kItems ? lane : 0);
    const uint64_t start_word = s_starts[my_word], kept_word = s_kept[my_word];
    const int start_before = s_starts_before[my_word] + before - 1;
    const int place = s_kept_before[my_word] + s_prefix;
    unsigned row[kItems];                                    // bit 31 as in s_row
    // starts at or before the lane: those below it in the word without its first bit, and the first bit
    auto group_by_bits = [&](int k) {
        const uint64_t word = lane_value(start_word, k);
        const int head = __builtin_amdgcn_readlane(start_before, k) + static_cast<int>(word & 1ull);
        return max(head + ballot_rank(word >> 1), 0);        // a slot before the first group is never used
    };
    if (by_bits && staged) {
#pragma unroll
        for (int k = 0; k < kItems; ++k) row[k] = s_row[group_by_bits(k)];
    } else {
#pragma unroll 1
        for (int k = 0; k < kItems; ++k) {
            unsigned found = 0u;
            if (!is_last || lane_value(kept_word, k) != 0ull) {      // the same for the whole wave; the last layer marks nobody
                int a = 0;
                if (by_bits) {
                    a = group_by_bits(k);
                } else {
                    const int e = static_cast<int>(base + mine + k * kWave);
                    int b = g_cnt;
                    while (b - a > 1) {
                        const int mid = (a + b) >> 1;
                        if (part_ptr[g_lo + mid] <= e) a = mid; else b = mid;
                    }
                }
                const int r = part2node[g_lo + a];
                found = static_cast<unsigned>(r) | (!is_last && in_mask<kBits>(src, r) ? 0x80000000u : 0u);
            }
#pragma unroll
            for (int j = 0; j < kItems; ++j) row[j] = j == k ? found : row[j];
        }
    }
    // ---- neighbours of marked rows
    if (!is_last) {
        // a vertex that already reads as marked is not stored again: hubs are neighbours of most rows
        constexpr int kMarks = kItems < 8 ? kItems : 8;
#pragma unroll
        for (int k0 = 0; k0 < kItems; k0 += kMarks) {
            bool want[kMarks];
            uint8_t seen[kMarks];
#pragma unroll
            for (int k = 0; k < kMarks; ++k) {
                const unsigned pos = static_cast<unsigned>(mine + (k0 + k) * kWave - owned_first);
                want[k] = row[k0 + k] >> 31 && pos < owned_slots && c[k0 + k] >= 0;
                seen[k] = ngh_mask[want[k] ? static_cast<unsigned>(c[k0 + k]) : 0u];      // no branch: all loads under way together
            }
#pragma unroll
            for (int k = 0; k < kMarks; ++k)
                if (want[k] && seen[k] == 0) ngh_mask[static_cast<unsigned>(c[k0 + k])] = 1;
        }
    }
    // ---- kept slots
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const uint64_t ballot = lane_value(kept_word, k);
        const unsigned to = __builtin_amdgcn_readlane(place, k), rank = static_cast<unsigned>(ballot_rank(ballot));
        if (__builtin_amdgcn_inverse_ballot_w64(ballot)) {
            const unsigned r = row[k] & 0x7fffffffu;
            (out_id + to)[rank] = static_cast<int>(r);
            (out_edge + to)[rank] = c[k];
            if (self_kept && static_cast<int>(r) == c[k]) self_kept[r] = 1;
        }
    }
    // ---- kept slots per row, and the marked rows themselves
    auto kept_before = [&](long long p) {                    // kept slots of the tile before slot base + p
        const int q = static_cast<int>(p < 0 ? 0 : p > kTile ? kTile : p);
        const int word = q >> 6;
        const int whole = s_kept_before[word];
        return (q & 63) ? whole + __popcll(s_kept[word] & ((1ull << (q & 63)) - 1ull)) : whole;
    };
    auto count_rows = [&](const Groups& g, int i0) {
        unsigned row[kBatch];
        if (staged) {
#pragma unroll
            for (int j = 0; j < kBatch; ++j) row[j] = s_row[min(i0 + j * kBlock + static_cast<int>(threadIdx.x), g_cnt - 1)];
        } else {
            load_rows(row, i0);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (i0 + j * kBlock >= g_cnt) break;             // the same for the whole workgroup
            const bool some = i0 + j * kBlock + static_cast<int>(threadIdx.x) < g_cnt;
            const int r = some ? static_cast<int>(row[j] & 0x7fffffffu) : -1;
            int n = some ? kept_before(g.to[j] - base) - kept_before(g.from[j] - base) : 0;
            const int left = __builtin_amdgcn_update_dpp(-2, r, kDppWaveShr1, 0xF, 0xF, false);
            n = wave_run_sum(n, __ballot(left != r));        // lane 0 starts a run
            if (left != r && n > 0) atomicAdd(node_degs + r, n);
            if (some && row[j] >> 31 && g.to[j] > g.from[j]) ngh_mask[r] = 1;
        }
    };
    count_rows(first, 0);
    for (int i0 = kBlock * kBatch; i0 < g_cnt; i0 += kBlock * kBatch) {
        Groups g;
        load_groups(g, i0);
        count_rows(g, i0);
    }
    // ---- zeros behind the kept slots of the whole input, written here and not by a pass of their own because they cost what
    // their bytes cost.  As many words as this tile drops slots, counted from the end, behind those of the tiles before it
    // (which dropped base - s_prefix slots).
    const long long end = length - (base - s_prefix);
    const long long from = end - (inside - s_kept_before[kWords]);
    zero_from(out_id, from, end, threadIdx.x, kBlock);
    zero_from(out_edge, from, end, threadIdx.x, kBlock);
}

// ---------------------------------------------------------------- the pass with everything a path needs around it
// Before: the source mask packed into bits, the scan state, the tiles' first groups, no row seen with its self-loop.
__global__ __launch_bounds__(256) void mark_path_init_kernel(const uint8_t* __restrict__ src_mask, int num_nodes, int words,
                                                             uint32_t* __restrict__ bits, uint32_t* __restrict__ self_kept,
                                                             const int* __restrict__ part_ptr, int num_parts, int num_tiles,
                                                             int* __restrict__ first, ScanState* st)
{
    const int i0 = blockIdx.x * 256 + threadIdx.x, stride = gridDim.x * 256;
    if (i0 == 0) *st = ScanState{};
    mark_tile_groups(part_ptr, num_parts, num_tiles, first, i0, stride);
    // a thread packs 4 bytes into 4 bits of a word, 8 lanes a word (vertices past the end count as unmarked)
    const bool quads = reinterpret_cast<uintptr_t>(src_mask) % 4 == 0;
    for (int q0 = blockIdx.x * 256; q0 < words * 8; q0 += stride) {
        const int q = q0 + static_cast<int>(threadIdx.x);
        unsigned nibble = 0u;
        if (q < words * 8) {
            const int v = q * 4;
            self_kept[q] = 0u;
            if (quads && v + 4 <= num_nodes) {
                nibble = nonzero_bytes(*reinterpret_cast<const uint32_t*>(src_mask + v));
            } else {
                for (int j = 0; j < 4; ++j)
                    if (v + j < num_nodes && src_mask[v + j]) nibble |= 1u << j;
            }
        }
        unsigned word = nibble << (4 * (threadIdx.x & 7));
        word |= __shfl_xor(word, 1, kWave);
        word |= __shfl_xor(word, 2, kWave);
        word |= __shfl_xor(word, 4, kWave);
        if ((threadIdx.x & 7) == 0 && q < words * 8) bits[q >> 3] = word;
    }
}

// After: the rows the path gathers, the rows with kept slots.
// Every vertex of the source mask whose self-loop is a slot is gathered; when that is all of them (graphs with
// self-loops, the usual case) the mask is the bitmap of the gathered rows and no pass over the kept slots is needed
// (0.58 ms for 126 M of them).  st->pad: [0] vertices of the mask, [1] not all of them kept their self-loop, [2] rows with
// kept slots.
// counts[1]: groups of at most group_size slots that the kept slots of the rows make (group_size 0: not counted).  Every
// workgroup ends in four atomics on one line (12 ns each, serial), so there are few of them and they are large.
constexpr int kFinishBlock = 1024, kFinishBlocks = 128;
__global__ __launch_bounds__(kFinishBlock) void mark_path_finish_kernel(const uint32_t* __restrict__ bits,
                                                                        const uint4* __restrict__ self_kept, int words,
                                                                        uint32_t* __restrict__ gathered,
                                                                        const int* __restrict__ node_degs, int num_nodes,
                                                                        int group_size, ScanState* st)
{
    constexpr int kWaves = kFinishBlock / kWave;
    __shared__ int s_sum[4][kWaves];
    const int i0 = blockIdx.x * kFinishBlock + threadIdx.x, stride = gridDim.x * kFinishBlock;
    int marked = 0, missing = 0, rows = 0, groups = 0;
    const unsigned gs = static_cast<unsigned>(max(group_size, 1));
    auto count_row = [&](int d) {
        rows += d != 0;
        groups += d > 0 ? static_cast<int>((static_cast<unsigned>(d) + gs - 1u) / gs) : 0;
    };
    for (int w = i0; w < words; w += stride) {
        const uint32_t b = bits[w];
        const uint4 lo = self_kept[2 * static_cast<size_t>(w)], hi = self_kept[2 * static_cast<size_t>(w) + 1];
        const uint32_t seen = nonzero_bytes(lo.x) | nonzero_bytes(lo.y) << 4 | nonzero_bytes(lo.z) << 8 |
                              nonzero_bytes(lo.w) << 12 | nonzero_bytes(hi.x) << 16 | nonzero_bytes(hi.y) << 20 |
                              nonzero_bytes(hi.z) << 24 | nonzero_bytes(hi.w) << 28;
        gathered[w] = b;
        marked += __popc(b);
        missing |= seen != b;
    }
    if (reinterpret_cast<uintptr_t>(node_degs) % 16 == 0) {
        const int4* quads = reinterpret_cast<const int4*>(node_degs);
#pragma unroll 4
        for (int v = i0; v < num_nodes / 4; v += stride) {
            const int4 d = quads[v];
            count_row(d.x); count_row(d.y); count_row(d.z); count_row(d.w);
        }
        if (i0 < num_nodes % 4) count_row(node_degs[num_nodes / 4 * 4 + i0]);
    } else {
        for (int v = i0; v < num_nodes; v += stride) count_row(node_degs[v]);
    }
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int sums[4] = {wave_inclusive_scan(marked), wave_inclusive_scan(missing), wave_inclusive_scan(rows), wave_inclusive_scan(groups)};
    if (lane == kWave - 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) s_sum[j][wave] = sums[j];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) sum += s_sum[threadIdx.x][w];
        int* const to[4] = {&st->pad[0], &st->pad[1], &st->pad[2], &st->counts[1]};
        if (sum && (threadIdx.x < 3 || group_size > 0)) atomicAdd(to[threadIdx.x], sum);
    }
}


// Zero both outputs from the compacted length (read on the device) to the end.
__global__ void zero_tail2_kernel(int* __restrict__ a, int* __restrict__ b, const int* __restrict__ d_start, int length)
{
    const long long i0 = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
    zero_from(a, *d_start, length, i0, stride);
    zero_from(b, *d_start, length, i0, stride);
}

// A workgroup per kTailWords consecutive words; those that lie before the start have nothing to do.  512 workgroups that
// stride over the array took 123 / 91 us for the two paths of R-MAT scale 22 (530 MB each), this 105 / 92.
constexpr int kTailWords = 16384;
__global__ __launch_bounds__(256) void zero_tail1_kernel(int* __restrict__ a, const int* __restrict__ d_start, int offset,
                                                         long long length)
{
    const long long first = static_cast<long long>(blockIdx.x) * kTailWords;
    zero_from(a, max(first, static_cast<long long>(*d_start) + offset), min(first + kTailWords, length), threadIdx.x, 256);
}

// ================================================================ counting
__global__ __launch_bounds__(256) void count_nonzero_kernel(const int* __restrict__ in, int length, int* __restrict__ d_count)
{
    int local = 0;
    const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
    for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < length; i += stride)
        local += in[i] != 0;
    add_block_count(local, d_count);
}

// ================================================================ distinct rows of a list
// Which of the rows 0 .. num_rows - 1 occur in list[0 .. length).  A byte per row is set with plain stores (every
// writer stores the same 1, so no order matters) and packed into bits afterwards.  A byte that already reads as set
// is not stored again: hub rows occur millions of times, and a stale copy in the vector cache only costs a store.
// Setting bits with atomics instead was bound by the serial updates of the hubs' words: 7.7 M entries over 2^20 rows
// 368 -> 40 us + 6 us for the packing, 126 M entries over 2^22 rows 947 -> 582 + 8 us.
__global__ __launch_bounds__(256) void mark_bytes_kernel(const int* __restrict__ list, long long length,
                                                         uint8_t* __restrict__ bytes, int* __restrict__ d_count)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *d_count = 0;       // for pack_bytes_kernel, which runs next
    const long long stride = static_cast<long long>(gridDim.x) * 256 * 4;
    const long long start = (static_cast<long long>(blockIdx.x) * 256 + threadIdx.x) * 4;
    const bool vec = reinterpret_cast<uintptr_t>(list) % 16 == 0;
    for (long long i = start; i < length; i += stride) {
        unsigned c[4];
        if (vec && i + 4 <= length) {
            const uint4 q = *reinterpret_cast<const uint4*>(list + i);
            c[0] = q.x; c[1] = q.y; c[2] = q.z; c[3] = q.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) c[j] = static_cast<unsigned>(list[i + j < length ? i + j : i]);
        }
        uint8_t seen[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) seen[j] = bytes[c[j]];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (!seen[j]) bytes[c[j]] = 1;
    }
}

// bitmap word w = bytes 32 w .. 32 w + 31 (the byte array is padded to whole words with zeros)
__global__ __launch_bounds__(256) void pack_bytes_kernel(const uint4* __restrict__ bytes, int words,
                                                         uint32_t* __restrict__ bitmap, int* __restrict__ d_count)
{
    const int w = blockIdx.x * 256 + threadIdx.x;
    unsigned bits = 0;
    if (w < words) {
        const uint4 lo = bytes[2 * static_cast<size_t>(w)], hi = bytes[2 * static_cast<size_t>(w) + 1];
        bits = nonzero_bytes(lo.x) | nonzero_bytes(lo.y) << 4 | nonzero_bytes(lo.z) << 8 | nonzero_bytes(lo.w) << 12 |
               nonzero_bytes(hi.x) << 16 | nonzero_bytes(hi.y) << 20 | nonzero_bytes(hi.z) << 24 | nonzero_bytes(hi.w) << 28;
        bitmap[w] = bits;
    }
    add_block_count(__popc(bits), d_count);
}

// The same without scratch memory: the bits are set with atomics in place (nothing waits for their result) and
// counted afterwards.
__global__ __launch_bounds__(256) void mark_bits_kernel(const int* __restrict__ list, long long length,
                                                        uint32_t* __restrict__ bitmap)
{
    const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
    for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < length; i += stride) {
        const unsigned c = static_cast<unsigned>(list[i]);
        const uint32_t bit = 1u << (c & 31);
        if ((bitmap[c >> 5] & bit) == 0) atomicOr(bitmap + (c >> 5), bit);
    }
}

__global__ __launch_bounds__(256) void count_bits_kernel(const uint32_t* __restrict__ bitmap, int words, int* __restrict__ d_count)
{
    int local = 0;
    for (int w = blockIdx.x * 256 + threadIdx.x; w < words; w += gridDim.x * 256) local += __popc(bitmap[w]);
    add_block_count(local, d_count);
}

// Degree histogram of get_ginfo (EPPGCN/GCNConv/EPPGCN.cpp:356-377): hist[0] = #(deg != 0),
// hist[3..9] = the seven buckets, the last one also taking deg <= 0 and deg >= 160.
__global__ __launch_bounds__(256) void ginfo_hist_kernel(const int* __restrict__ node_deg, int length, int* __restrict__ hist)
{
    int local[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
    for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < length; i += stride) {
        const int deg = node_deg[i];
        local[0] += deg != 0;
        int b = 7;
        if (deg >= 1 && deg < 5) b = 1;
        else if (deg >= 5 && deg < 10) b = 2;
        else if (deg >= 10 && deg < 20) b = 3;
        else if (deg >= 20 && deg < 40) b = 4;
        else if (deg >= 40 && deg < 80) b = 5;
        else if (deg >= 80 && deg < 160) b = 6;
#pragma unroll
        for (int k = 1; k < 8; ++k) local[k] += b == k;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        int s = local[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, kWave);
        if ((threadIdx.x & (kWave - 1)) == 0 && s) atomicAdd(hist + (k == 0 ? 0 : k + 2), s);
    }
}

// ================================================================ group splitting
// Vertex i with g_i slots (g_i = kept degree, or CSR degree) yields q_i = ceil(g_i/ps)
// groups; group j of vertex i starts at G_i + j*ps where G_i is the exclusive sum
// of g.  One look-back scan carries (sum q, sum g) packed as q*2^31 + g over tiles of kSplitTile vertices; vertex
// (round r, thread t) of a tile is r * kSplitBlock + t, so that degrees are read and groups written with neighbouring
// lanes on neighbouring words; the (round, wave) sums are scanned by one wave.  The tile's groups are written in two ways:
// a vertex with at most kSmallGroups groups by the thread that owns it, every other vertex - collected on a list in LDS -
// by a whole wave, 64 groups per step, so a hub with a hundred thousand groups costs its tile a longer loop, not one
// thread a longer life.  The tile with the hubs is the last to finish (the first 2048 vertices of an R-MAT graph of scale
// 22 have 200 thousand groups): 16 waves write it.  4 waves, with 8 consecutive vertices per thread: 0.19 ms for the forward
// groups of that graph against 0.07, and 84 against 31 us at scale 20.
constexpr int kSplitBlock = 1024;
constexpr int kSplitRounds = 2;
constexpr int kSplitTile = kSplitBlock * kSplitRounds;
constexpr int kSplitWaves = kSplitBlock / kWave;
constexpr int kSmallGroups = 4;     // groups per vertex up to which the owning thread writes them itself
static_assert(kSplitRounds * kSplitWaves <= kWave, "one wave scans the (round, wave) sums of a tile");

template <bool kFromRowPtr>
__global__ __launch_bounds__(kSplitBlock) void split_groups_kernel(
    const int* __restrict__ src, int num_nodes, int part_size, int* __restrict__ part_ptr_out,
    int* __restrict__ part2node_out, long long capacity, long long rows_capacity, int num_tiles, ScanState* st, uint64_t* desc,
    unsigned mode)
{
    __shared__ int s_tile;
    __shared__ uint64_t s_sum[kSplitRounds * kSplitWaves];
    __shared__ int s_big_first[kSplitTile], s_big_start[kSplitTile], s_big_groups[kSplitTile], s_big_vertex[kSplitTile];
    __shared__ int s_big_count;
    if (threadIdx.x == 0) s_big_count = 0;
    const int tile = acquire_tile(st, &s_tile);
    if (tile >= num_tiles) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long base = static_cast<long long>(tile) * kSplitTile;

    int q[kSplitRounds];
    uint64_t at[kSplitRounds];             // (groups, slots) before the vertex
#pragma unroll
    for (int r = 0; r < kSplitRounds; ++r) {
        const long long i = base + r * kSplitBlock + threadIdx.x;
        int g = 0;
        if (i < num_nodes) g = kFromRowPtr ? src[i + 1] - src[i] : src[i];
        g = g > 0 ? g : 0;
        q[r] = (g + part_size - 1) / part_size;
        const uint64_t mine = (static_cast<uint64_t>(q[r]) << 31) | static_cast<uint64_t>(g);
        const uint64_t incl = wave_inclusive_scan_u64(mine);
        at[r] = incl - mine;
        if (lane == kWave - 1) s_sum[r * kSplitWaves + wave] = incl;
    }
    const int g_first = kFromRowPtr ? src[0] : 0;
    __syncthreads();
    if (wave == 0) {
        const uint64_t mine = lane < kSplitRounds * kSplitWaves ? s_sum[lane] : 0ull;
        const uint64_t incl = wave_inclusive_scan_u64(mine);
        const uint64_t total = static_cast<uint64_t>(__shfl(static_cast<long long>(incl), kWave - 1, kWave));
        const uint64_t excl = tile_lookback(desc, st, tile, total, mode);
        if (lane < kSplitRounds * kSplitWaves) s_sum[lane] = excl + incl - mine;
        if (tile == num_tiles - 1 && lane == 0) {
            const uint64_t all = excl + total;
            const int total_q = static_cast<int>(all >> 31);
            const int total_g = static_cast<int>(all & 0x7fffffffull);
            st->counts[0] = total_q;
            st->counts[1] = total_g;
            if (total_q < capacity) part_ptr_out[total_q] = total_g + g_first;
            if (static_cast<long long>(total_q) + 1 > capacity || (part2node_out && total_q > rows_capacity)) st->overflow = 1;
        }
    }
    __syncthreads();
    auto write_group = [&](long long dst, int start, int vertex) {
        if (dst < capacity) {
            part_ptr_out[dst] = start;
            if (part2node_out && dst < rows_capacity) part2node_out[dst] = vertex;
        }
    };
#pragma unroll
    for (int r = 0; r < kSplitRounds; ++r) {
        const uint64_t before = s_sum[r * kSplitWaves + wave] + at[r];
        const int first = static_cast<int>(before >> 31);
        const int start = static_cast<int>(before & 0x7fffffffull) + g_first;
        const int vertex = static_cast<int>(base) + r * kSplitBlock + static_cast<int>(threadIdx.x);
        if (q[r] > kSmallGroups) {
            const int b = atomicAdd(&s_big_count, 1);
            s_big_first[b] = first;
            s_big_start[b] = start;
            s_big_groups[b] = q[r];
            s_big_vertex[b] = vertex;
        } else {
#pragma unroll
            for (int k = 0; k < kSmallGroups; ++k)
                if (k < q[r]) write_group(static_cast<long long>(first) + k, start + k * part_size, vertex);
        }
    }
    __syncthreads();
    const int big = s_big_count;
    for (int b = wave; b < big; b += kSplitWaves) {
        const int groups = s_big_groups[b];
        const long long first = s_big_first[b];
        const int start = s_big_start[b], vertex = s_big_vertex[b];
        // The first 64 groups like any others, the others of a hub in loops without bounds checks, all of them its one wave's.  With
        // the checks in a single loop its speed hung on where the code before it let it start in the instruction cache (the split of
        // R-MAT scale 21 into groups of one slot 1018 us, 1145 after that code had shrunk; now 824).
        if (lane < groups) write_group(first + lane, start + lane * part_size, vertex);
        if (groups <= kWave) continue;
        const int ptrs = static_cast<int>(min(static_cast<long long>(groups), max(capacity - first, 0ll)));
        const int rows = part2node_out ? static_cast<int>(min(static_cast<long long>(ptrs), max(rows_capacity - first, 0ll))) : 0;
        for (int k = lane + kWave; k < ptrs; k += kWave) part_ptr_out[first + k] = start + k * part_size;
        for (int k = lane + kWave; k < rows; k += kWave) part2node_out[first + k] = vertex;
    }
}

// ================================================================ host launchers
__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t* __restrict__ p, size_t head, size_t vecs, size_t words)
{
    // [0, head) scalar words up to the first 16-byte boundary, then `vecs` uint4, then the rest
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    const size_t tid = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    uint4* v = reinterpret_cast<uint4*>(p + head);
    // non-temporal: the zeros are not read back before the kernel that follows has filled the caches
    typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
    const uintx4 zero = {0u, 0u, 0u, 0u};
    for (size_t i = tid; i < vecs; i += stride) __builtin_nontemporal_store(zero, reinterpret_cast<uintx4*>(v) + i);
    const size_t tail = head + 4 * vecs;
    if (tid < head) p[tid] = 0u;
    if (tid < words - tail) p[tail + tid] = 0u;
}

int launch_zero_words(void* p, size_t words, hipStream_t stream)
{
    if (words == 0) return kOk;
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    size_t head = ((16 - a % 16) % 16) / 4;
    if (head > words) head = words;
    const size_t vecs = (words - head) / 4;
    // one vector per thread: 528 MB at 6.8 TB/s, against 5.5 with 2^14 workgroups that stride over it
    size_t blocks = (vecs + 255) / 256;
    if (blocks > (1u << 23)) blocks = 1u << 23;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(zero_words_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream,
                       static_cast<uint32_t*>(p), head, vecs, words);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

// out[num_rows, dim]: one thread per vector of VW floats; a row whose bit in `skip` is set is left alone.
// Index: unsigned when the vector count fits in 32 bits (the row of a vector is then a 32-bit division).
template <int VW, class Index>
__global__ __launch_bounds__(256) void zero_rows_unless_kernel(float* __restrict__ out, const uint32_t* __restrict__ skip,
                                                               Index total_vecs, Index vecs_per_row)
{
    typedef float fvec __attribute__((ext_vector_type(VW)));
    const Index stride = static_cast<Index>(gridDim.x) * blockDim.x;
    for (Index i = static_cast<Index>(blockIdx.x) * blockDim.x + threadIdx.x; i < total_vecs; i += stride) {
        const Index r = i / vecs_per_row;
        if (!((skip[r >> 5] >> (r & 31)) & 1u)) {
            if constexpr (VW == 1) {
                __builtin_nontemporal_store(0.f, out + i);
            } else {
                fvec z = {};
                __builtin_nontemporal_store(z, reinterpret_cast<fvec*>(out) + i);
            }
        }
        if (total_vecs - i <= stride) break;      // the next index would run past the end (and could wrap)
    }
}

// The same with the work found by whole waves: a wave looks at 64 rows at a time, collects those whose bit
// is clear (usually few: the rows of several groups or of none) and clears them VW floats per lane, so
// the cost follows the rows that are cleared instead of the size of the matrix.
template <int VW>
__global__ __launch_bounds__(256) void zero_listed_rows_kernel(float* __restrict__ out, const uint32_t* __restrict__ skip,
                                                               unsigned num_rows, unsigned vecs_per_row)
{
    typedef float fvec __attribute__((ext_vector_type(VW)));
    __shared__ int lists[4][kWave];
    int* list = lists[threadIdx.x / kWave];
    const unsigned lane = lane_id();
    const unsigned waves = gridDim.x * 4u;
    const unsigned blocks64 = (num_rows + 63u) / 64u;
    for (unsigned b = blockIdx.x * 4u + threadIdx.x / kWave; b < blocks64; b += waves) {
        const unsigned r = b * 64u + lane;
        const bool wanted = r < num_rows && ((skip[r >> 5] >> (r & 31)) & 1u) == 0;
        const unsigned count = compact_wanted_rows(list, r, wanted);
        const unsigned total = count * vecs_per_row;
        for (unsigned t = lane; t < total; t += kWave) {
            const unsigned k = t / vecs_per_row;
            const size_t at = static_cast<size_t>(list[k]) * vecs_per_row + (t - k * vecs_per_row);
            if constexpr (VW == 1) {
                __builtin_nontemporal_store(0.f, out + at);
            } else {
                fvec z = {};
                __builtin_nontemporal_store(z, reinterpret_cast<fvec*>(out) + at);
            }
        }
    }
}

static std::atomic<bool> g_force_wide_index{false};
bool force_wide_index() { return g_force_wide_index.load(); }
void set_force_wide_index(bool on) { g_force_wide_index.store(on); }

int launch_zero_rows_unless(float* out, const uint32_t* skip, long long num_rows, int dim, hipStream_t stream)
{
    if (num_rows <= 0 || dim <= 0) return kOk;
    const uintptr_t a = reinterpret_cast<uintptr_t>(out);
    const int vw = (dim % 4 == 0 && a % 16 == 0) ? 4 : (dim % 2 == 0 && a % 8 == 0) ? 2 : 1;
    const int vecs_per_row = dim / vw;
    if (num_rows < (1ll << 31) && !force_wide_index()) {
        long long blocks = (num_rows + 255) / 256;           // one wave per 64 rows
        if (blocks > 256 * 16) blocks = 256 * 16;
        const dim3 grid(static_cast<unsigned>(blocks)), block(256);
        const unsigned n = static_cast<unsigned>(num_rows), v = static_cast<unsigned>(vecs_per_row);
        if (vw == 4) hipLaunchKernelGGL(zero_listed_rows_kernel<4>, grid, block, 0, stream, out, skip, n, v);
        else if (vw == 2) hipLaunchKernelGGL(zero_listed_rows_kernel<2>, grid, block, 0, stream, out, skip, n, v);
        else hipLaunchKernelGGL(zero_listed_rows_kernel<1>, grid, block, 0, stream, out, skip, n, v);
    } else {
        // any size: one thread per vector of the matrix
        const unsigned long long total = static_cast<unsigned long long>(num_rows) * vecs_per_row;
        unsigned long long blocks = (total + 255) / 256;
        if (blocks > 256 * 64) blocks = 256 * 64;
        const dim3 grid(static_cast<unsigned>(blocks)), block(256);
        const unsigned long long v = static_cast<unsigned long long>(vecs_per_row);
        if (vw == 4) hipLaunchKernelGGL((zero_rows_unless_kernel<4, unsigned long long>), grid, block, 0, stream, out, skip, total, v);
        else if (vw == 2) hipLaunchKernelGGL((zero_rows_unless_kernel<2, unsigned long long>), grid, block, 0, stream, out, skip, total, v);
        else hipLaunchKernelGGL((zero_rows_unless_kernel<1, unsigned long long>), grid, block, 0, stream, out, skip, total, v);
    }
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

size_t scan_workspace_bytes(long long length, int tile)
{
    const long long tiles = (length + tile - 1) / tile;
    return sizeof(ScanState) + sizeof(uint64_t) * static_cast<size_t>(tiles > 0 ? tiles : 1);
}

size_t compact_workspace_bytes(long long length) { return scan_workspace_bytes(length, kCompactTile); }
size_t split_workspace_bytes(long long num_nodes) { return scan_workspace_bytes(num_nodes, kSplitTile); }

// Workgroups of zero_tail2_kernel, which clears what lies behind a length that only the device knows: two per CU (528 MB at
// 5.9 TB/s with 512 workgroups that stride over it, at 4.3 with 2048).
constexpr int kTailBlocks = 512;
static unsigned tail_blocks(long long length)
{
    const long long blocks = (length + 1023) / 1024;
    return static_cast<unsigned>(blocks > kTailBlocks ? kTailBlocks : blocks < 1 ? 1 : blocks);
}

static int init_scan(void* workspace, int num_tiles, hipStream_t stream)
{
    ScanState* st = static_cast<ScanState*>(workspace);
    uint64_t* desc = reinterpret_cast<uint64_t*>(st + 1);
    const int n = num_tiles > 0 ? num_tiles : 1;
    hipLaunchKernelGGL(scan_init_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, st, desc, num_tiles);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

int launch_mask_forward(const int* part2node, const int* part_ptr, const int* col, const uint8_t* src_mask,
                        uint8_t* ngh_mask, int* back_edge_mask, int* node_degs, int num_parts,
                        long long num_edges, int is_last, hipStream_t stream)
{
    (void)num_edges;
    if (num_parts == 0) return kOk;
    const long long groups_per_block = static_cast<long long>(kWave) * kMaskWaves;
    const unsigned grid = static_cast<unsigned>((num_parts + groups_per_block - 1) / groups_per_block);
    hipLaunchKernelGGL(mask_forward_kernel, dim3(grid), dim3(kMaskBlock), 0, stream, part2node, part_ptr, col, src_mask,
                       ngh_mask, back_edge_mask, node_degs, num_parts, is_last);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

// Results land in the ScanState at the head of the workspace: counts[0] = kept length.
int launch_compact_mask(const int* in_id, int* out_id, const int* in_edge, int* out_edge, long long length,
                        void* workspace, hipStream_t stream)
{
    ScanState* st = static_cast<ScanState*>(workspace);
    uint64_t* desc = reinterpret_cast<uint64_t*>(st + 1);
    const int num_tiles = static_cast<int>((length + kCompactMaskTile - 1) / kCompactMaskTile);
    if (int rc = init_scan(workspace, num_tiles, stream)) return rc;
    if (num_tiles > 0) {
        hipLaunchKernelGGL(compact_mask_kernel, dim3(num_tiles), dim3(kCompactBlock), 0, stream, in_id, in_edge,
                           out_id, out_edge, static_cast<int>(length), num_tiles, st, desc, scan_mode());
        EPPGCN_HIP(hipGetLastError());
        hipLaunchKernelGGL(zero_tail2_kernel, dim3(tail_blocks(length)), dim3(256), 0, stream, out_id, out_edge, st->counts,
                           static_cast<int>(length));
        EPPGCN_HIP(hipGetLastError());
    }
    return kOk;
}

// ---- allocation-free compaction: the scan workspace is the file-scope device array `scratch`
long long static_compact_max_length() { return kStaticCompactMaxLength; }

// Device address of `scratch` on the current device, looked up once per device (every GPU holds
// its own copy of the array at its own address).
static int static_compact_scratch(void** out)
{
    constexpr int kMaxDevices = 64;
    static std::mutex lock;
    static void* address[kMaxDevices] = {nullptr};
    int device = 0;
    EPPGCN_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) {
        set_error("static scratch: device ordinal " + std::to_string(device) + " is outside 0..63");
        return kErrInvalidArgument;
    }
    std::lock_guard<std::mutex> guard(lock);
    if (!address[device]) {
        void* p = nullptr;
        EPPGCN_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p || reinterpret_cast<uintptr_t>(p) % 8 != 0) {
            set_error("static scratch: hipGetSymbolAddress returned an unusable address");
            return kErrHip;
        }
        address[device] = p;
    }
    *out = address[device];
    return kOk;
}

// The scratch address for the status call (and the look-up of the address outside a graph capture).
int static_compact_workspace(void** out) { return static_compact_scratch(out); }

// compact_mask_kernel over the static scratch; *workspace_out receives the scratch address (its
// ScanState holds the kept length once the stream has run).  The scan state and the descriptors of
// the tiles this call uses are cleared by init_scan's fill kernel on every call: the array keeps
// the previous call's contents.
int launch_compact_mask_static(const int* in_id, int* out_id, const int* in_edge, int* out_edge, long long length,
                               void** workspace_out, hipStream_t stream)
{
    static_assert(kStaticCompactTile == kCompactMaskTile && kStaticCompactMaxLength % kCompactMaskTile == 0 &&
                      kStaticCompactScratchBytes == sizeof(ScanState) + 8 * (kStaticCompactMaxLength / kCompactMaskTile),
                  "the static scratch holds the scan state and one descriptor per tile of compact_mask_kernel");
    void* ws = nullptr;
    if (int rc = static_compact_scratch(&ws)) return rc;
    *workspace_out = ws;
    return launch_compact_mask(in_id, out_id, in_edge, out_edge, length, ws, stream);
}

// Workspace of the marking pass behind its ScanState: one bit per slot, a count and the first group of every tile, and
// for launch_mark_path the bit map of the source mask and one byte per vertex (its self-loop was kept), in whole words.
struct MarkLayout {
    size_t kept, counts, first, bits, self_kept, total;
    int num_tiles, words;
};
static MarkLayout mark_layout(long long length, long long num_nodes)
{
    MarkLayout l;
    l.num_tiles = static_cast<int>((length + kMarkTile - 1) / kMarkTile);
    l.words = static_cast<int>((num_nodes + 31) / 32);
    l.kept = sizeof(ScanState);
    l.counts = l.kept + static_cast<size_t>(l.num_tiles) * (kMarkTile / 8);
    l.first = l.counts + 4 * static_cast<size_t>(l.num_tiles);
    l.bits = (l.first + 4 * (static_cast<size_t>(l.num_tiles) + 1) + 15) / 16 * 16;
    l.self_kept = (l.bits + 4 * static_cast<size_t>(l.words) + 15) / 16 * 16;
    l.total = l.self_kept + 32 * static_cast<size_t>(l.words);
    return l;
}
size_t mark_compact_workspace_bytes(long long length) { return mark_layout(length < 0 ? 0 : length, 0).total; }
size_t mark_path_workspace_bytes(long long length, long long num_nodes) { return mark_layout(length, num_nodes).total; }
uint8_t* mark_path_scratch(void* workspace, long long length, long long num_nodes)
{
    return static_cast<uint8_t*>(workspace) + mark_layout(length, num_nodes).self_kept;
}

template <bool kBits>
static int launch_mark_pass(const int* part2node, const int* part_ptr, const int* col, const void* src, uint8_t* ngh_mask,
                            int* node_degs, int* out_id, int* out_edge, uint8_t* self_kept, int num_parts, long long length,
                            int is_last, const MarkLayout& l, char* workspace, hipStream_t stream)
{
    ScanState* st = reinterpret_cast<ScanState*>(workspace);
    unsigned long long* kept = reinterpret_cast<unsigned long long*>(workspace + l.kept);
    int* counts = reinterpret_cast<int*>(workspace + l.counts);
    const int* first = reinterpret_cast<const int*>(workspace + l.first);
    const dim3 grid(l.num_tiles);
    const int len = static_cast<int>(length);
    hipLaunchKernelGGL(keep_slots_kernel<kBits>, grid, dim3(kKeepBlock), 0, stream, part_ptr, col, src, num_parts, len, kept, counts);
    EPPGCN_HIP(hipGetLastError());
#define EPPGCN_PLACE(BLOCK_, SCANNED_)                                                                                    \
    hipLaunchKernelGGL((place_slots_kernel<BLOCK_, SCANNED_, kBits>), grid, dim3(BLOCK_), 0, stream, part2node, part_ptr,  \
                       col, src, ngh_mask, node_degs, out_id, out_edge, self_kept, num_parts, len, l.num_tiles, is_last,    \
                       first, kept, counts, st)
    // place_slots walks a tile from barrier to barrier.  1024 threads do that fastest as long as the chip holds all tiles at once
    // (two workgroups on a CU: 512 tiles), beyond that smaller workgroups hide each other's waits better.  The kernel, us, with
    // 1024 / 512 / 256 threads: 27 tiles 12 / 13 / -, 2253 tiles - / 41 / 46, 32 thousand tiles, the mean of two layers, - / 413 /
    // 392; a whole marking: 564 tiles 37 / 33 / 38, 4395 tiles 143 / 123 / 119, 10 thousand tiles 315 / 274 / 275.
    if (l.num_tiles >= kMarkScannedTiles) {
        hipLaunchKernelGGL(scan_counts_kernel, dim3(1), dim3(1024), 0, stream, counts, l.num_tiles);
        EPPGCN_HIP(hipGetLastError());
        EPPGCN_PLACE(256, true);
    } else if (l.num_tiles > 512) {
        EPPGCN_PLACE(512, false);
    } else {
        EPPGCN_PLACE(1024, false);
    }
    EPPGCN_HIP(hipGetLastError());
#undef EPPGCN_PLACE
    return kOk;
}

// Results land in the ScanState at the head of the workspace: counts[0] = kept length.
int launch_mark_compact(const int* part2node, const int* part_ptr, const int* col, const uint8_t* src_mask,
                        uint8_t* ngh_mask, int* node_degs, int* out_id, int* out_edge, int num_parts,
                        long long length, int is_last, void* workspace, hipStream_t stream)
{
    const MarkLayout l = mark_layout(length, 0);
    char* base = static_cast<char*>(workspace);
    if (num_parts == 0 || l.num_tiles == 0) {
        if (int rc = init_scan(workspace, 0, stream)) return rc;
        if (length > 0) {
            if (int rc = launch_zero_words(out_id, static_cast<size_t>(length), stream)) return rc;
            if (int rc = launch_zero_words(out_edge, static_cast<size_t>(length), stream)) return rc;
        }
        return kOk;
    }
    ScanState* st = static_cast<ScanState*>(workspace);
    const int blocks = num_parts / 1024 + 1 < 4096 ? num_parts / 1024 + 1 : 4096;
    hipLaunchKernelGGL(tile_groups_kernel, dim3(blocks), dim3(256), 0, stream, part_ptr, num_parts,
                       l.num_tiles, reinterpret_cast<int*>(base + l.first), st);
    EPPGCN_HIP(hipGetLastError());
    if (int rc = launch_mark_pass<false>(part2node, part_ptr, col, src_mask, ngh_mask, node_degs, out_id, out_edge, nullptr,
                                         num_parts, length, is_last, l, base, stream))
        return rc;
    return kOk;
}

// launch_mark_compact with the rows of the path counted and its gathered rows marked; num_parts, length, num_nodes > 0.
// Results land in the ScanState at the head of the workspace (16-byte aligned): counts[0] = kept length, counts[1] and pad as
// mark_path_finish_kernel says.
int launch_mark_path(const int* part2node, const int* part_ptr, const int* col, const uint8_t* src_mask,
                     uint8_t* ngh_mask, int* node_degs, int* out_id, int* out_edge, uint32_t* gathered, int num_parts,
                     long long length, int num_nodes, int is_last, int group_size, void* workspace, hipStream_t stream)
{
    const MarkLayout l = mark_layout(length, num_nodes);
    char* base = static_cast<char*>(workspace);
    ScanState* st = static_cast<ScanState*>(workspace);
    uint32_t* bits = reinterpret_cast<uint32_t*>(base + l.bits);
    uint8_t* self_kept = reinterpret_cast<uint8_t*>(base + l.self_kept);
    const int most = l.words * 8 > num_parts / 4 ? l.words * 8 : num_parts / 4;
    const int init_blocks = most / 256 + 1 < 4096 ? most / 256 + 1 : 4096;
    hipLaunchKernelGGL(mark_path_init_kernel, dim3(init_blocks), dim3(256), 0, stream, src_mask, num_nodes, l.words, bits,
                       reinterpret_cast<uint32_t*>(self_kept), part_ptr, num_parts, l.num_tiles,
                       reinterpret_cast<int*>(base + l.first), st);
    EPPGCN_HIP(hipGetLastError());
    if (int rc = launch_mark_pass<true>(part2node, part_ptr, col, bits, ngh_mask, node_degs, out_id, out_edge, self_kept,
                                        num_parts, length, is_last, l, base, stream))
        return rc;
    const int count_blocks = num_nodes / 16384 + 1 < kFinishBlocks ? num_nodes / 16384 + 1 : kFinishBlocks;
    hipLaunchKernelGGL(mark_path_finish_kernel, dim3(count_blocks), dim3(kFinishBlock), 0, stream, bits,
                       reinterpret_cast<const uint4*>(self_kept), l.words, gathered, node_degs, num_nodes, group_size,
                       st);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

// Before a split of kept degrees: the scan state, and the whole array of group pointers cleared.  With groups of the usual
// size they are a few hundredths of the entries, so clearing what they overwrite costs less than a launch behind the split
// that first has to know their end: path preparation at R-MAT scale 22 3954 -> 3908 us, at 19 717 vertices 1.5 % less.  Groups
// of one to three slots can fill most of a large array: there the tail is cleared afterwards (zero_tail1_kernel).
// A split, us, cleared before / behind, with every slot kept (groups of 1 / 2 / 3 fill 78 / 42 / 29 % of the entries):
//   0.6 M entries  groups of 1, 3, 4 slots: 27.2 / 29.1, 13.3 / 15.4, 7.9 / 10.1      1.3 M  28.3 / 29.9, 14.3 / 16.1, 9.1 / 10.9
//   5 M            35.7 / 34.9, 20.8 / 21.7, 14.7 / 15.7      161 M  608 / 546, 355 / 349, 272 / 279, of 32 slots 224 / 243
// and with a tenth of the slots kept, 161 M: 262 / 287, 238 / 269, 227 / 260.  So both lines are on the cautious side: groups
// of one slot are even at 4 M entries, and below that, and with few slots kept, clearing before is up to 2 us (a tenth) faster
// also for groups of less than four slots, which clear behind from 1 M entries on.
constexpr int kClearFirstPartSize = 4;
constexpr long long kClearFirstEntries = 1 << 20;
__global__ __launch_bounds__(256) void split_init_kernel(ScanState* st, uint64_t* desc, int num_tiles, int* __restrict__ p,
                                                         size_t head, size_t vecs, size_t words)
{
    const size_t tid = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x, stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = tid; i < static_cast<size_t>(num_tiles); i += stride) desc[i] = kTileEmpty;
    if (tid == 0) {
        st->counter = 0;
        st->error = 0;
        st->counts[0] = 0;
        st->counts[1] = 0;
        st->overflow = 0;
    }
    typedef int intx4 __attribute__((ext_vector_type(4)));
    const intx4 zero = {0, 0, 0, 0};
    intx4* v = reinterpret_cast<intx4*>(p + head);
    for (size_t i = tid; i < vecs; i += stride) __builtin_nontemporal_store(zero, v + i);
    const size_t tail = head + 4 * vecs;
    if (tid < head) p[tid] = 0;
    if (tid < words - tail) p[tail + tid] = 0;
}

// counts[0] = number of groups, counts[1] = number of slots covered.
// part2node_out (may be NULL for degrees): the vertex of every group, rows_capacity entries
int launch_split(bool from_row_ptr, const int* src, int num_nodes, int part_size, int* part_ptr_out,
                 int* part2node_out, long long capacity, long long rows_capacity, bool zero_tail, void* workspace,
                 hipStream_t stream)
{
    ScanState* st = static_cast<ScanState*>(workspace);
    uint64_t* desc = reinterpret_cast<uint64_t*>(st + 1);
    const int num_tiles = (num_nodes + kSplitTile - 1) / kSplitTile;
    const bool tail_after = zero_tail && num_tiles > 0 && part_size < kClearFirstPartSize && capacity > kClearFirstEntries;
    if ((zero_tail && !tail_after) || num_tiles == 0) {
        const size_t words = capacity <= 0 ? 0 : zero_tail ? static_cast<size_t>(capacity) : 1;
        const size_t misaligned = reinterpret_cast<uintptr_t>(part_ptr_out) / 4 % 4;
        const size_t head = misaligned && 4 - misaligned < words ? 4 - misaligned : misaligned ? words : 0;
        const size_t vecs = (words - head) / 4;
        size_t blocks = (vecs + 255) / 256;
        if (blocks > (1u << 23)) blocks = 1u << 23;
        if (blocks < 1) blocks = 1;
        hipLaunchKernelGGL(split_init_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, st, desc, num_tiles,
                           part_ptr_out, head, vecs, words);
        EPPGCN_HIP(hipGetLastError());
        if (num_tiles == 0) return kOk;
    } else {
        if (int rc = init_scan(workspace, num_tiles, stream)) return rc;
    }
    if (from_row_ptr)
        hipLaunchKernelGGL((split_groups_kernel<true>), dim3(num_tiles), dim3(kSplitBlock), 0, stream, src, num_nodes,
                           part_size, part_ptr_out, part2node_out, capacity, rows_capacity, num_tiles, st, desc, scan_mode());
    else
        hipLaunchKernelGGL((split_groups_kernel<false>), dim3(num_tiles), dim3(kSplitBlock), 0, stream, src, num_nodes,
                           part_size, part_ptr_out, part2node_out, capacity, rows_capacity, num_tiles, st, desc, scan_mode());
    EPPGCN_HIP(hipGetLastError());
    if (tail_after) {
        hipLaunchKernelGGL(zero_tail1_kernel, dim3(static_cast<unsigned>((capacity + kTailWords - 1) / kTailWords)), dim3(256), 0,
                           stream, part_ptr_out, st->counts, 1, capacity);
        EPPGCN_HIP(hipGetLastError());
    }
    return kOk;
}

// The first bytes of up to kStateList records on the device, kStateBytes each, into host memory that the device can write:
// one launch and one wait for all of them, where a copy and a wait for each took 20 to 25 us a record.
struct StateList { const uint32_t* from[kStateList]; };
__global__ __launch_bounds__(256) void gather_states_kernel(StateList list, int count, uint32_t* __restrict__ to)
{
    constexpr int kWords = kStateBytes / 4;
    for (int i = threadIdx.x; i < count * kWords; i += 256) to[i] = list.from[i / kWords][i % kWords];
}

int launch_gather_states(const void* const* states, int count, void* host, hipStream_t stream)
{
    uint32_t* to = static_cast<uint32_t*>(host);
    for (int at = 0; at < count; at += kStateList) {
        StateList list = {};
        const int some = count - at < kStateList ? count - at : kStateList;
        for (int i = 0; i < some; ++i) list.from[i] = static_cast<const uint32_t*>(states[at + i]);
        hipLaunchKernelGGL(gather_states_kernel, dim3(1), dim3(256), 0, stream, list, some,
                           to + static_cast<size_t>(at) * (kStateBytes / 4));
        EPPGCN_HIP(hipGetLastError());
    }
    return kOk;
}

int launch_count_nonzero(const int* in, long long length, int* d_count, hipStream_t stream)
{
    if (int rc = launch_zero_words(d_count, 1, stream)) return rc;
    if (length == 0) return kOk;
    long long blocks = (length + 4095) / 4096;
    if (blocks > 512) blocks = 512;
    hipLaunchKernelGGL(count_nonzero_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, in,
                       static_cast<int>(length), d_count);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

// bytes of scratch with which launch_mark_listed_rows works without atomics: one per row, whole bitmap words
size_t mark_listed_rows_scratch_bytes(long long num_rows) { return static_cast<size_t>((num_rows + 31) / 32) * 32; }

// scratch: nullptr or mark_listed_rows_scratch_bytes(num_rows), 16-byte aligned
int launch_mark_listed_rows(const int* list, long long length, long long num_rows, uint32_t* bitmap, int* d_count,
                            uint8_t* scratch, hipStream_t stream)
{
    const int words = static_cast<int>((num_rows + 31) / 32);
    if (length == 0 || words == 0) {
        if (int rc = launch_zero_words(bitmap, static_cast<size_t>(words), stream)) return rc;
        return launch_zero_words(d_count, 1, stream);
    }
    if (scratch) {
        if (int rc = launch_zero_words(scratch, static_cast<size_t>(words) * 8, stream)) return rc;
        long long blocks = (length + 1023) / 1024;
        if (blocks > 2048) blocks = 2048;
        hipLaunchKernelGGL(mark_bytes_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, list, length,
                           scratch, d_count);
        EPPGCN_HIP(hipGetLastError());
        hipLaunchKernelGGL(pack_bytes_kernel, dim3((words + 255) / 256), dim3(256), 0, stream,
                           reinterpret_cast<const uint4*>(scratch), words, bitmap, d_count);
        EPPGCN_HIP(hipGetLastError());
        return kOk;
    }
    if (int rc = launch_zero_words(bitmap, static_cast<size_t>(words), stream)) return rc;
    if (int rc = launch_zero_words(d_count, 1, stream)) return rc;
    long long blocks = (length + 1023) / 1024;
    if (blocks > 512) blocks = 512;
    hipLaunchKernelGGL(mark_bits_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, list, length, bitmap);
    EPPGCN_HIP(hipGetLastError());
    long long count_blocks = (words + 1023) / 1024;
    if (count_blocks > 512) count_blocks = 512;
    hipLaunchKernelGGL(count_bits_kernel, dim3(static_cast<unsigned>(count_blocks)), dim3(256), 0, stream, bitmap, words, d_count);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

int launch_ginfo_hist(const int* node_deg, long long length, int* d_hist10, hipStream_t stream)
{
    if (int rc = launch_zero_words(d_hist10, 10, stream)) return rc;
    if (length == 0) return kOk;
    long long blocks = (length + 1023) / 1024;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(ginfo_hist_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, node_deg,
                       static_cast<int>(length), d_hist10);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

}  // namespace eppgcn

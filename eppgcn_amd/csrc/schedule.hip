// Column-blocked execution plan for the aggregation kernels.
//
// The aggregation gathers feature rows at random; in CSR row order the rows gathered at any
// moment are spread over the whole table and two thirds of the gathers go to HBM.  A plan is a
// copy of the groups re-ordered by the column block of their first slot (blocks of 2^shift
// vertices, original order inside a block): the waves in flight then work on one window of
// columns whose rows are served from L2.  The plan holds everything the kernel reads per group
// in processing order, so that all of it streams:
//
//     ptr[P+1]   slot offsets into `col`            row[P]    row of the group
//     flags[P]   bit0 the row has groups before this one (original order), bit1 after it,
//                bit2 this group continues the previous plan entry (same row, next original
//                index), bit3 the next plan entry continues this one
//     col[S]     column ids, group by group in plan order
//     single[ceil(N/32)]  bit r set: row r has exactly one group and the group is not empty; the
//                kernel writes such a row with one plain store, so the output clear can skip it
//
// Stream form (for stream.hip).  Consecutive plan entries that continue one another form a piece (a stretch
// of slots of one row); the last slot of every piece carries bit 31 in col[], col[] is padded to a multiple
// of 512 slots with an id behind every table row (N rounded up to a multiple of 4096), and
//     erow[e]    row of piece e when the stream kernel can write it with one store (the piece is all of its row
//                and lies inside one chunk, the 512 slots of a workgroup), otherwise bit 31 | index of the partial
//                sum it leaves
//     cev[c]     pieces that end before slot 32 c; bit 31 when slot 32 c continues a piece
//     wtail[w]   index of the partial sum for what chunk w still holds at its last slot, or -1
//     touched    one bit per vertex: the row has at least one slot
//     frow/fptr  rows that have partial sums and the range of each; the partial sums are numbered row by row,
//                inside a row those of its piece ends, then those of the chunks' tails, each in the caller's group order
//                (the stream's too when the columns of a row ascend), so that summing a range in order gives the
//                same bits every run
// and a header with the counts.  A plan with empty groups gets no stream form (header.valid = 0).
//
// The re-ordering changes no result, only which groups run together.  It depends on the graph
// and the groups alone: a caller builds it once and passes it to every aggregation call.
//
// How a plan is built (launch_build_plan), all on the device and without a host read-back:
//   plan_init      clears the scan states, the two row bitmaps and the header
//   plan_keys      per group, in the caller's order: row, adjacency, sort key, the digit counts of the first radix pass
//   radix passes   stable least-significant-digit sort of (key, group index), the last pass moves the groups' records; none
//                  for a plan in one block
//   plan_order     per plan entry: one look-back scan over (slots, piece ends) gives the slot offsets and the piece
//                  numbers together; writes ptr / row / flags and the extent of every piece
//   plan_fill      per 2048 slots: the column copy with the piece-end flags, cev, wtail preset
//   plan_partials  per group, in the caller's order again: which pieces leave partial sums, numbered by two
//                  look-back scans side by side.  A row's groups are neighbours in this order, so the numbers come out
//                  row by row without sorting the pieces by row (a three-pass sort of 8 M candidates before)
//   plan_targets   writes erow / wtail from those numbers and completes the header
// Every kernel streams its arrays once; what used to be 46 launches, four of them radix passes over 8 M keys, is 9.  R-MAT
// scale 22, both paths and the forward groups of a two-layer run (7.8 + 5.9 + 1.7 M groups, 132 + 126 + 13 M slots):
// 6.0 -> 1.65 ms for the three plans; scale 20 (8.8 + 7.3 + 0.9 M slots): 1.3 -> 0.30 ms.
#include <atomic>
#include <cstring>

#include "common.hpp"

namespace eppgcn {

static size_t align256(size_t x) { return (x + 255) / 256 * 256; }

// ---------------------------------------------------------------- look-back scan (radix offsets)
// Exclusive prefix sum of `in[0..n)` into `out[0..n]` (out[n] = total): single pass, decoupled
// look-back over tiles of 2048.
constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems;

__global__ __launch_bounds__(kScanBlock) void exclusive_scan_kernel(const int* __restrict__ in, int* __restrict__ out,
                                                                   int n, int num_tiles, ScanState* st, uint64_t* desc, unsigned mode)
{
    __shared__ int s_tile;
    __shared__ int s_wave[kScanBlock / kWave];
    __shared__ int s_excl;
    const int tile = acquire_tile(st, &s_tile);
    if (tile >= num_tiles) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long base = static_cast<long long>(tile) * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    int sum = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        v[j] = base + j < n ? in[base + j] : 0;
        sum += v[j];
    }
    const int incl = wave_inclusive_scan(sum);
    if (lane == kWave - 1) s_wave[wave] = incl;
    __syncthreads();
    int wave_excl = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kScanBlock / kWave; ++w) {
        if (w < wave) wave_excl += s_wave[w];
        total += s_wave[w];
    }
    if (wave == 0) {
        const uint64_t excl = tile_lookback(desc, st, tile, static_cast<uint64_t>(total), mode);
        if (lane == 0) s_excl = static_cast<int>(excl);
    }
    __syncthreads();
    int run = s_excl + wave_excl + incl - sum;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        if (base + j < n) out[base + j] = run;
        run += v[j];
    }
    if (tile == num_tiles - 1 && threadIdx.x == kScanBlock - 1) out[n] = run;
}

// ---------------------------------------------------------------- stable radix sort of (key, index) pairs
// One pass sorts by the digit (key >> shift) & (digits - 1), digits = 2^bits <= 256, and keeps the order of equal
// digits, so passes from the least significant digit upwards sort by the whole key, equal keys staying in index order.
// A tile is kSortTile consecutive elements, element (round r, thread t) of tile T being T * kSortTile + r * 256 + t, so
// that (round, wave, lane) order is index order.
//   plan_keys_kernel / radix_hist_kernel   hist[d * tiles + T] = elements of tile T with digit d
//   exclusive_scan_kernel over hist (digit-major): where (digit d, tile T) starts in the output
//   radix_scatter_kernel  rank of an element among the equal digits of its wave from one ballot per digit bit,
//                         counts per (round, wave, digit) in LDS, prefix over (round, wave) per digit
constexpr int kSortBlock = 256;
constexpr int kSortRounds = 8;
constexpr int kSortTile = kSortBlock * kSortRounds;
constexpr int kDigits = 256;

__global__ __launch_bounds__(kSortBlock) void radix_hist_kernel(const unsigned* __restrict__ keys, int n, int shift,
                                                                int digits, int num_tiles, int* __restrict__ hist)
{
    __shared__ int s_hist[kDigits];
    s_hist[threadIdx.x] = 0;
    __syncthreads();
    const long long base = static_cast<long long>(blockIdx.x) * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const long long i = base + r * kSortBlock + threadIdx.x;
        if (i < n) atomicAdd(&s_hist[(keys[i] >> shift) & (digits - 1)], 1);
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < digits)
        hist[static_cast<long long>(threadIdx.x) * num_tiles + blockIdx.x] = s_hist[threadIdx.x];
}

// vals_in == nullptr: the value of element i is i (first pass).  The last pass (rec_out) takes the records of the groups along
// and leaves where each went in vals_out; nobody reads its keys.  A tile is 2048 groups in the caller's order, which go to one
// run of neighbours per digit: this is the direction in which the records move in whole lines.  plan_order_kernel, which has
// to take neighbours in sorted order, looked its groups up in four arrays before, each in lines of its own.  The builds of
// R-MAT scale 22 (7.8 + 5.9 M groups sorted), us: plan_order 431 -> 191, this kernel 49 -> 118, plan_partials 215 -> 249 (it
// reads the places); scale 20: 83 -> 53, 12 -> 23, 58 -> 64.
__global__ __launch_bounds__(kSortBlock) void radix_scatter_kernel(const unsigned* __restrict__ keys_in,
                                                                   const int* __restrict__ vals_in,
                                                                   unsigned* __restrict__ keys_out,
                                                                   int* __restrict__ vals_out, int n, int shift, int bits,
                                                                   int num_tiles, const int* __restrict__ offsets,
                                                                   const int4* __restrict__ rec_in, int4* __restrict__ rec_out)
{
    constexpr int kWaves = kSortBlock / kWave;
    __shared__ int s_count[kSortRounds * kWaves][kDigits];      // per (round, wave): elements of each digit
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int digits = 1 << bits;
    for (int i = threadIdx.x; i < kSortRounds * kWaves * digits; i += kSortBlock)
        s_count[i >> bits][i & (digits - 1)] = 0;
    __syncthreads();
    const long long base = static_cast<long long>(blockIdx.x) * kSortTile;
    unsigned key[kSortRounds];
    int rank[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const long long i = base + r * kSortBlock + threadIdx.x;
        key[r] = i < n ? keys_in[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const bool valid = base + r * kSortBlock + threadIdx.x < n;
        const unsigned d = (key[r] >> shift) & (digits - 1);
        // lanes of the wave holding the same digit: intersect the ballots of the digit's bits
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
            const uint64_t set = __ballot(((d >> b) & 1u) != 0);
            peers &= ((d >> b) & 1u) ? set : ~set;
        }
        rank[r] = __popcll(peers & ((1ull << lane) - 1ull));
        if (valid && rank[r] == 0) s_count[r * kWaves + wave][d] = __popcll(peers);
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < digits) {
        // thread d: exclusive prefix of digit d over the (round, wave) pairs, on top of the tile's global offset
        int run = offsets[static_cast<long long>(threadIdx.x) * num_tiles + blockIdx.x];
#pragma unroll
        for (int q = 0; q < kSortRounds * kWaves; ++q) {
            const int c = s_count[q][threadIdx.x];
            s_count[q][threadIdx.x] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const long long i = base + r * kSortBlock + threadIdx.x;
        if (i < n) {
            const unsigned d = (key[r] >> shift) & (digits - 1);
            const int dst = s_count[r * kWaves + wave][d] + rank[r];
            const int val = vals_in ? vals_in[i] : static_cast<int>(i);
            if (dst >= 0 && dst < n && val >= 0 && val < n) {   // false only after a stalled scan
                if (rec_out) {
                    rec_out[dst] = rec_in[val];
                    vals_out[val] = dst;
                } else {
                    keys_out[dst] = key[r];
                    vals_out[dst] = val;
                }
            }
        }
    }
}

// ---------------------------------------------------------------- plan kernels
struct PlanScans {            // states of the look-back scans of one build, inside the workspace
    ScanState* sort;          // radix offsets
    ScanState* order;         // plan_order
    ScanState* partials;      // plan_partials (two descriptor arrays: ends and tails, rows)
    uint64_t *sort_desc, *order_desc, *ends_desc, *rows_desc;
    int sort_tiles, order_tiles;
};

// one launch clears everything a build counts on being clear
__global__ __launch_bounds__(256) void plan_init_kernel(StreamHeader* h, PlanScans sc, uint32_t* __restrict__ single,
                                                        uint32_t* __restrict__ touched, int words, int num_parts,
                                                        int num_slots, int num_nodes, int generation,
                                                        const ScanState* upstream)
{
    const int stride = gridDim.x * blockDim.x;
    const int i0 = blockIdx.x * blockDim.x + threadIdx.x;
    for (int i = i0; i < words; i += stride) { single[i] = 0u; touched[i] = 0u; }
    for (int i = i0; i < sc.sort_tiles; i += stride) sc.sort_desc[i] = kTileEmpty;
    for (int i = i0; i < sc.order_tiles; i += stride) {
        sc.order_desc[i] = kTileEmpty;
        sc.ends_desc[i] = kTileEmpty;
        sc.rows_desc[i] = kTileEmpty;
    }
    if (i0 == 0) {
        *sc.sort = ScanState{};
        // groups of a split that stalled are not to be read, and groups that cover other slots than the caller's are not the
        // path's: every kernel that would read them ends at this flag
        if (upstream && (upstream->error || upstream->overflow || upstream->counts[0] != num_parts || upstream->counts[1] != num_slots))
            sc.sort->error = 1;
        *sc.order = ScanState{};
        *sc.partials = ScanState{};
        StreamHeader z = {};
        z.empty_rows = num_nodes;
        z.magic = kPlanMagic;
        z.generation = generation;
        z.num_parts = num_parts;
        z.num_nodes = num_nodes;
        z.num_slots = num_slots;
        *h = z;
    }
}

// Sets bit (row & 31) of touched[row >> 5] for the lanes with `set`, and of single[row >> 5] for those with `alone` too: the
// lanes of a wave whose rows share a word (rows ascend along the groups, so they are neighbours) combine their bits first,
// one atomic per run.  A row's bit is counted in its first lane, so the bits of a run are distinct and their sum is their union;
// rows that do not ascend are set one by one.  One atomic per group was most of the classification kernel before (0.7 ms per run
// at R-MAT scale 22); combining the bits in six shuffle steps per map cost plan_keys 22 of 401 us more than these sums.
__device__ __forceinline__ void or_row_bits(uint32_t* __restrict__ touched, uint32_t* __restrict__ single, int row, bool set,
                                            bool alone)
{
    const int mine = set ? row : -1;
    const int left = __builtin_amdgcn_update_dpp(-1, mine, kDppWaveShr1, 0xF, 0xF, false);
    const int bit = static_cast<int>(1u << (row & 31));
    if (__any(set && left > row)) {
        if (set) atomicOr(touched + (row >> 5), static_cast<uint32_t>(bit));
        if (set && alone) atomicOr(single + (row >> 5), static_cast<uint32_t>(bit));
        return;
    }
    const uint64_t heads = __ballot(left >> 5 != mine >> 5) | 1ull;
    const uint32_t all = static_cast<uint32_t>(wave_run_sum(set && left != row ? bit : 0, heads));
    const uint32_t some = static_cast<uint32_t>(wave_run_sum(set && left != row && alone ? bit : 0, heads));
    if ((heads >> lane_id()) & 1ull) {
        if (all) atomicOr(touched + (row >> 5), all);
        if (some) atomicOr(single + (row >> 5), some);
    }
}

// What plan_order_kernel needs of a group, 16 bytes that the sort moves: first slot, slots, row, number; bit 31 of the first two:
// the row has groups before / after this one.
__device__ __forceinline__ int4 pack_group(int beg, int size, int row, int p, bool before, bool after)
{
    return make_int4(beg | (before ? static_cast<int>(kStreamFlag) : 0), size | (after ? static_cast<int>(kStreamFlag) : 0), row, p);
}

// Per group p: rowp[p] (0 for an empty group; rowp == nullptr: part2node is that array), rec[p] (pack_group; nullptr: nothing is
// sorted), info[p] = bit0 the row has groups before this one, bit1 after it, bit2 the group has slots; the row bitmaps; the sort
// key and the digit counts of the first radix pass (keys == nullptr: the plan keeps the caller's order).
// Sort key of group p: the column block of its first slot, except that all groups of a short row
// (at most `keep_slots` slots in at most kMaxRowWalk groups) share the key of the row's first group:
// such a row stays together in the plan, is summed in registers and written once with plain stores,
// instead of leaving one partial sum per column block (measured at group size 31: the partial sums of rows with 2..16
// groups cost more than the L2 hits of their later groups save; the bound is in slots because a row's gathers, not its
// groups, are what a block can speed up: with groups of 4-8 slots a bound in groups spread rows of 40 slots and lost up
// to 2x at 256 columns).
// The walk to the ends of a row stops as soon as the row cannot be short any more: with the usual group sizes that is
// after two or three groups.  It runs over pointers and rows in LDS, those of the tile and of the 64 groups on either side of it
// (a step was a round trip to memory, one round of groups after the other: 48 us for the 705 tiles of R-MAT scale 20, all of
// which run at once; with the sorted path of that scale 81 -> 52 us, with 256 threads 69, with 1024 48 but 6 % slower at scale
// 22), and the columns that decide the keys are loaded together.  What is left at scale 22 (7.8 M groups 202 -> 190 us) is one
// cache line of `col` per group, and one of `ids` where the rows are looked up there: 5.9 M groups of a path 347 us with ids, 172
// with the rows that the split left (eppgcn_split_and_plan).
constexpr int kMaxRowWalk = 64;
constexpr int kKeysBlock = 512;
constexpr int kKeysRounds = kSortTile / kKeysBlock;
static_assert(kSortTile % kKeysBlock == 0 && kKeysBlock >= kDigits, "group (round r, thread t) of a tile is r * 512 + t; a thread per digit");
__global__ __launch_bounds__(kKeysBlock) void plan_keys_kernel(
    const int* __restrict__ part_ptr, const int* __restrict__ col, const int* __restrict__ part2node,
    const int* __restrict__ ids, int num_parts, int num_nodes, int shift, int keep_slots, int classes, int digits,
    int num_tiles, unsigned* __restrict__ keys, int* __restrict__ hist, int* __restrict__ rowp, uint8_t* __restrict__ info,
    int4* __restrict__ rec, uint32_t* __restrict__ single, uint32_t* __restrict__ touched, StreamHeader* __restrict__ h, const ScanState* sort_state)
{
    constexpr int kHalo = kMaxRowWalk;                  // groups of the neighbouring tiles that a walk can reach
    constexpr int kStaged = kSortTile + 2 * kHalo;
    __shared__ int s_ptr[kStaged + 1];                  // [i]: group base - kHalo + i
    __shared__ int s_row[kStaged];
    __shared__ int s_hist[kDigits];
    if (sort_state->error) return;
    if (threadIdx.x < kDigits) s_hist[threadIdx.x] = 0;
    const int base = static_cast<int>(static_cast<long long>(blockIdx.x) * kSortTile);      // < num_parts
    const long long origin = static_cast<long long>(base) - kHalo;
    for (int i = threadIdx.x; i <= kStaged; i += kKeysBlock) {
        const long long g = min(max(origin + i, 0ll), static_cast<long long>(num_parts));
        s_ptr[i] = part_ptr[g];
        if (part2node && i < kStaged) s_row[i] = part2node[min(g, static_cast<long long>(num_parts) - 1)];
    }
    __syncthreads();
    if (!part2node) {
        for (int i = threadIdx.x; i < kStaged; i += kKeysBlock)
            s_row[i] = s_ptr[i + 1] > s_ptr[i] ? ids[s_ptr[i]] : 0;
        __syncthreads();
    }
    int at[kKeysRounds], cls[kKeysRounds];              // slot whose column decides the key (-1: an empty group's), length class
#pragma unroll
    for (int r = 0; r < kKeysRounds; ++r) {
        const int i = kHalo + r * kKeysBlock + static_cast<int>(threadIdx.x);
        const long long pl = origin + i;
        const int p = static_cast<int>(pl);
        const bool have = pl < num_parts;
        const int beg = s_ptr[i], end = s_ptr[i + 1];
        const bool some = have && end > beg;
        const int row = some ? s_row[i] : 0;
        int before = -1, after = -1;
        if (some) {
            if (part2node) {
                if (p > 0) before = s_row[i - 1];
                if (p + 1 < num_parts) after = s_row[i + 1];
            } else {
                if (beg > 0) before = ids[beg - 1];
                if (p + 1 < num_parts) after = ids[end];
            }
        }
        const bool prev = some && before == row, next = some && after == row;
        if (have) {
            if (rowp) rowp[p] = row;
            info[p] = static_cast<uint8_t>((prev ? 1 : 0) | (next ? 2 : 0) | (some ? 4 : 0));
            if (rec) rec[p] = pack_group(beg, some ? end - beg : 0, row, p, prev, next);
            if (!some) h->empty_groups = 1;
        }
        const bool in_range = some && row >= 0 && row < num_nodes;
        or_row_bits(touched, single, row, in_range, !prev && !next);
        at[r] = -1;
        cls[r] = 0;
        if (!keys || !some) continue;
        auto same_row = [&](int j) { return s_ptr[j + 1] > s_ptr[j] && s_row[j] == row; };
        const int lo = base < kHalo ? kHalo - base : 0;                                         // group 0
        const int hi = static_cast<int>(min(static_cast<long long>(kStaged), num_parts - origin));      // behind the last group
        int start = i, last = i;
        bool short_row = keep_slots > 0 && end - beg <= keep_slots;
        int first_slot = beg, past = end;
        while (short_row && start > lo && same_row(start - 1)) {
            first_slot = s_ptr[--start];
            short_row = past - first_slot <= keep_slots && i - start < kMaxRowWalk;
        }
        while (short_row && last + 1 < hi && same_row(last + 1)) {
            past = s_ptr[++last + 1];
            short_row = past - first_slot <= keep_slots && last - start < kMaxRowWalk;
        }
        at[r] = short_row ? first_slot : beg;
        // second key: length class of a row that is a single group (a class = one gather step of 8
        // slots), so that the groups a wave works on in one round take the same number of steps;
        // rows of several groups consist of full groups but for the last one: class 3
        cls[r] = (short_row && start == last) ? min(3, (end - beg - 1) >> 3) : 3;
    }
    if (!keys) return;
    int first_col[kKeysRounds];
#pragma unroll
    for (int r = 0; r < kKeysRounds; ++r) first_col[r] = at[r] >= 0 ? col[at[r]] : 0;
#pragma unroll
    for (int r = 0; r < kKeysRounds; ++r) {
        const long long p = static_cast<long long>(base) + r * kKeysBlock + threadIdx.x;
        if (p >= num_parts) continue;
        unsigned key = static_cast<unsigned>(first_col[r]) >> shift;
        if (classes) key = (key << 2) | static_cast<unsigned>(cls[r]);
        keys[p] = key;
        atomicAdd(&s_hist[key & (digits - 1)], 1);
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < digits)
        hist[static_cast<long long>(threadIdx.x) * num_tiles + blockIdx.x] = s_hist[threadIdx.x];
}

// Tiles of the two scans over the groups: entry (round r, thread t) of tile T is T * kPlanTile + r * 512 + t, so that every
// array is read and written with full-width accesses and (round, wave, lane) order is entry order; the 64 (round, wave)
// sums of a tile are scanned by one wave.  8 consecutive entries per thread instead: 0.63
// and 0.26 ms for the two kernels over 15.4 M groups, against 0.45 and 0.22.  (The tile ids of a look-back
// scan come from one device counter at 12 ns each: tiles of 4096 keep that below 25 us for 8 M groups.)
constexpr int kPlanBlock = 512;
constexpr int kPlanItems = 8;
constexpr int kPlanTile = kPlanBlock * kPlanItems;
constexpr int kPlanWaves = kPlanBlock / kWave;
static_assert(kPlanItems * kPlanWaves == kWave, "one wave scans the (round, wave) sums of a tile");
constexpr int kFillTile = 2048;            // slots a workgroup of plan_fill_kernel writes
static_assert(kFillTile % kStreamWave == 0 && kFillTile % kStreamChunk == 0, "cev and wtail entries belong to one fill tile");

// Plan entry q holds the group of rec[q] (rec == nullptr: group q).  One scan carries (slots, piece ends) packed as
// ends * 2^31 + slots.  Piece e: extent[e] = its first slot | bit 31 when the row has groups before it, and its last
// slot; erow[e] = its row, event_at[q] = e for the entry q that ends it and -1 for every other entry.
// tile_q[t] = the plan entry that holds slot t * kFillTile.
__global__ __launch_bounds__(kPlanBlock) void plan_order_kernel(
    const int* __restrict__ part_ptr, const int4* __restrict__ rec, const int* __restrict__ rowp,
    const uint8_t* __restrict__ info, int num_parts, int num_slots, int num_tiles, PlanView plan, StreamView sv,
    int* __restrict__ src, int* __restrict__ ends_before, int2* __restrict__ extent,
    int* __restrict__ event_at, int* __restrict__ tile_q, ScanState* st, uint64_t* desc, unsigned mode, const ScanState* sort_state)
{
    __shared__ int s_tile;
    __shared__ uint64_t s_sum[kPlanItems * kPlanWaves];
    if (sort_state->error) return;
    const int tile = acquire_tile(st, &s_tile);
    if (tile >= num_tiles) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long q0 = static_cast<long long>(tile) * kPlanTile + threadIdx.x;
    int p[kPlanItems], side[kPlanItems];      // group of the entry; that of its neighbour in another wave (-1: none)
    int beg[kPlanItems], size[kPlanItems], row[kPlanItems];
    unsigned f[kPlanItems];                   // bit 0: the row has groups before this one, 1: after it, 2: slots
    auto side_of = [&](long long q) {         // entry of the neighbour in another wave
        return lane == 0 ? q - 1 : lane == kWave - 1 ? q + 1 : -1;
    };
    if (rec) {
        int4 g[kPlanItems];
#pragma unroll
        for (int r = 0; r < kPlanItems; ++r) {
            const long long q = q0 + r * kPlanBlock, n = side_of(q);
            g[r] = q < num_parts ? rec[q] : make_int4(0, 0, 0, -1);
            side[r] = n >= 0 && n < num_parts ? rec[n].w : -1;
        }
#pragma unroll
        for (int r = 0; r < kPlanItems; ++r) {
            p[r] = g[r].w;
            beg[r] = g[r].x & kStreamIdMask;
            size[r] = g[r].y & kStreamIdMask;
            row[r] = g[r].z;
            f[r] = (g[r].x < 0 ? 1u : 0u) | (g[r].y < 0 ? 2u : 0u) | (size[r] > 0 ? 4u : 0u);
        }
    } else {
#pragma unroll
        for (int r = 0; r < kPlanItems; ++r) {
            const long long q = q0 + r * kPlanBlock, n = side_of(q);
            const bool have = q < num_parts;
            const int g = static_cast<int>(have ? q : 0);
            p[r] = have ? g : -1;
            side[r] = n >= 0 && n < num_parts ? static_cast<int>(n) : -1;
            beg[r] = have ? part_ptr[g] : 0;
            size[r] = have ? max(part_ptr[g + 1] - beg[r], 0) : 0;
            row[r] = have ? rowp[g] : 0;
            f[r] = have ? info[g] : 0u;
        }
    }
    int at[kPlanItems], eb[kPlanItems];
    unsigned is_end = 0u;
#pragma unroll
    for (int r = 0; r < kPlanItems; ++r) {
        const int up = __shfl_up(p[r], 1, kWave), down = __shfl_down(p[r], 1, kWave);
        const int left = lane == 0 ? side[r] : up, right = lane == kWave - 1 ? side[r] : down;
        const bool joins_left = (f[r] & 1u) && left >= 0 && left == p[r] - 1;
        const bool joins_right = (f[r] & 2u) && right >= 0 && right == p[r] + 1;
        const bool ends = (f[r] & 4u) && !joins_right;
        f[r] = (f[r] & 3u) | (joins_left ? 4u : 0u) | (joins_right ? 8u : 0u);
        is_end |= ends ? 1u << r : 0u;
        const uint64_t ballot = __ballot(ends);
        const int incl = wave_inclusive_scan(size[r]);
        at[r] = incl - size[r];
        eb[r] = ballot_rank(ballot);
        if (lane == kWave - 1) s_sum[r * kPlanWaves + wave] = (static_cast<uint64_t>(__popcll(ballot)) << 31) + static_cast<uint64_t>(incl);
    }
    __syncthreads();
    if (wave == 0) {
        const uint64_t mine = s_sum[lane];
        const uint64_t incl = wave_inclusive_scan_u64(mine);
        const uint64_t total = static_cast<uint64_t>(__shfl(static_cast<long long>(incl), kWave - 1, kWave));
        const uint64_t excl = tile_lookback(desc, st, tile, total, mode);
        s_sum[lane] = excl + incl - mine;
        if (tile == num_tiles - 1 && lane == 0) {
            const uint64_t all = excl + total;
            plan.ptr[num_parts] = static_cast<int>(all & 0x7fffffffull);
            sv.header->num_events = min(static_cast<int>(all >> 31), num_parts);
            const int fill_tiles = static_cast<int>((static_cast<long long>(num_slots) + kFillTile - 1) / kFillTile);
            for (int t = static_cast<int>(((all & 0x7fffffffull) + kFillTile - 1) / kFillTile); t < fill_tiles; ++t)
                tile_q[t] = num_parts - 1;              // slots the caller counted and no group covers
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPlanItems; ++r) {
        if (p[r] < 0) continue;
        const int q = static_cast<int>(q0) + r * kPlanBlock;
        const uint64_t before = s_sum[r * kPlanWaves + wave];
        const int slot = at[r] + static_cast<int>(before & 0x7fffffffull);
        const int e = eb[r] + static_cast<int>(before >> 31);
        const bool ends = (is_end >> r) & 1u;
        plan.ptr[q] = slot;
        plan.row[q] = row[r];
        plan.flags[q] = static_cast<uint8_t>(f[r]);
        src[q] = beg[r];
        ends_before[q] = e;
        event_at[q] = ends ? e : -1;
        if (size[r] == 0) continue;
        if ((f[r] & 4u) == 0 && e < num_parts) extent[e].x = slot | ((f[r] & 1u) ? static_cast<int>(kStreamFlag) : 0);
        if (ends && e < num_parts) {
            extent[e].y = slot + size[r] - 1;
            sv.erow[e] = row[r];
        }
        for (long long t = (static_cast<long long>(slot) + kFillTile - 1) / kFillTile;
             t * kFillTile < min(static_cast<long long>(slot) + size[r], static_cast<long long>(num_slots)); ++t)
            tile_q[t] = q;
    }
}

// A workgroup writes kFillTile consecutive slots of plan.col: the plan entry (and so the source) of a slot is a prefix
// population count over a bit map of the entries' starts in LDS, loads and stores are coalesced whatever the group
// lengths are (a team of 8 lanes per group before: 0.52 -> 0.34 ms for 132 M slots, 1.06 GB read and written).
__global__ __launch_bounds__(256) void plan_fill_kernel(const int* __restrict__ col, PlanView plan, StreamView sv,
                                                       const int* __restrict__ src, const int* __restrict__ ends_before,
                                                       const int* __restrict__ tile_q, int num_parts, int num_slots,
                                                       int padded_slots, int num_nodes, int num_fill_tiles, PlanScans sc)
{
    constexpr int kItems = kFillTile / 256;
    constexpr int kWords = kFillTile / 64;
    __shared__ unsigned long long s_start[kWords];      // bit i: an entry starts at slot base + i (i > 0)
    __shared__ unsigned long long s_last[kWords];       // bit i: slot base + i is the last of a piece
    __shared__ int s_before[kWords];                    // entry starts before each word
    __shared__ int s_delta[kFillTile + 1];              // source slot - plan slot of every entry of the tile
    if (sc.sort->error || sc.order->error) return;      // the offsets are not to be trusted; the plan is refused
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int base = blockIdx.x * kFillTile;
    const int covered = min(plan.ptr[num_parts], num_slots);      // slots behind the groups' own gather nothing, as the padding
    const int q_lo = tile_q[blockIdx.x];
    const int q_hi = static_cast<int>(blockIdx.x) + 1 < num_fill_tiles ? tile_q[blockIdx.x + 1] : num_parts - 1;
    const int count = q_hi - q_lo + 1;
    const bool by_bits = sv.header->empty_groups == 0 && count <= kFillTile + 1;
    if (threadIdx.x < kWords) { s_start[threadIdx.x] = 0ull; s_last[threadIdx.x] = 0ull; }
    __syncthreads();
    for (int i = threadIdx.x; i < count; i += 256) {
        const int q = q_lo + i;
        const int a = plan.ptr[q], b = plan.ptr[q + 1];
        if (by_bits) s_delta[i] = src[q] - a;
        const int s = a - base, l = b - 1 - base;
        if (i > 0 && s > 0 && s < kFillTile) atomicOr(&s_start[s >> 6], 1ull << (s & 63));
        if (b > a && (plan.flags[q] & 8) == 0 && l >= 0 && l < kFillTile) atomicOr(&s_last[l >> 6], 1ull << (l & 63));
    }
    __syncthreads();
    if (wave == 0) {
        const int pc = lane < kWords ? __popcll(s_start[lane]) : 0;
        const int incl = wave_inclusive_scan(pc);
        if (lane < kWords) s_before[lane] = incl - pc;
    }
    __syncthreads();
    // plan entry of slot base + i, relative to q_lo
    auto owner = [&](int i) -> int {
        if (by_bits) {
            const unsigned long long upto = (i & 63) == 63 ? ~0ull : (2ull << (i & 63)) - 1ull;
            return s_before[i >> 6] + __popcll(s_start[i >> 6] & upto);
        }
        int a = 0, b = count;                           // empty groups: the last entry that starts at or before the slot
        while (b - a > 1) {
            const int mid = (a + b) >> 1;
            if (plan.ptr[q_lo + mid] <= base + i) a = mid; else b = mid;
        }
        return a;
    };
    int v[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int i = k * 256 + static_cast<int>(threadIdx.x);
        // "gathers nothing": an id whose row lies behind every table, in swizzled row order too
        v[k] = static_cast<int>(swizzle_padded_rows(num_nodes));
        if (base + i < covered) {
            const int o = owner(i);
            const int delta = by_bits ? s_delta[o] : src[q_lo + o] - plan.ptr[q_lo + o];
            v[k] = __builtin_nontemporal_load(col + base + i + delta);
        }
    }
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int i = k * 256 + static_cast<int>(threadIdx.x);
        const bool flagged = (s_last[i >> 6] >> (i & 63)) & 1ull;
        if (base + i < padded_slots)
            __builtin_nontemporal_store(v[k] | (flagged ? static_cast<int>(kStreamFlag) : 0), plan.col + base + i);
    }
    if (threadIdx.x < kFillTile / kStreamWave) {
        const int w = base / kStreamWave + threadIdx.x;
        if (w < padded_slots / kStreamWave) sv.wtail[w] = -1;
    }
    const bool closing = static_cast<int>(blockIdx.x) + 1 == num_fill_tiles;       // writes the entry behind the last slot too
    if (threadIdx.x <= kFillTile / kStreamChunk) {
        const int i = static_cast<int>(threadIdx.x) * kStreamChunk;
        const long long pos = static_cast<long long>(base) + i;      // one tile past 2^31 - 1 for the last tile of the largest plan
        const bool mine = i < kFillTile ? pos < padded_slots || (closing && pos == padded_slots) : closing && pos == padded_slots;
        if (mine) {
            int e = sv.header->num_events;
            bool inside = false;
            if (pos < covered) {
                const int q = q_lo + owner(i);
                e = ends_before[q];
                inside = pos > 0 && (plan.ptr[q] < pos || (plan.flags[q] & 4) != 0);
            }
            sv.cev[pos / kStreamChunk] = e | (inside ? static_cast<int>(kStreamFlag) : 0);
        }
    }
}

// Which pieces leave partial sums, and how many: a piece that is not all of its row, or that crosses from one chunk of
// 512 slots into the next, leaves one at its end, and one more per chunk boundary it crosses (what that chunk still holds
// at its last slot).  Group p (in the caller's order; plan entry place[p], nullptr: p) speaks for the piece it ends.  Two scans
// run side by side, wave 0's over (tails, ends) packed as tails * 2^31 + ends, wave 1's over (rows with slots, rows with
// partial sums).
// The partial sums of row j of the fix list are numbered ends first, then tails: its range starts at ends + tails before
// its first group.  fix_of[p] = j or -1; ends_at / tails_at[p] the counts before p; ends0 / tails0[j] those before row j.
__global__ __launch_bounds__(kPlanBlock) void plan_partials_kernel(
    const int* __restrict__ rowp, const uint8_t* __restrict__ info, const int* __restrict__ place,
    const int* __restrict__ event_at, int* __restrict__ event_of, const int2* __restrict__ extent,
    int num_parts, int num_nodes, int num_tiles,
    StreamView sv, int* __restrict__ fix_of, int* __restrict__ ends_at, int* __restrict__ tails_at,
    int* __restrict__ ends0, int* __restrict__ tails0, int* __restrict__ ends_total, PlanScans sc, unsigned mode)
{
    __shared__ int s_tile;
    __shared__ uint64_t s_sum[2][kPlanItems * kPlanWaves];
    if (sc.sort->error || sc.order->error || sv.header->empty_groups) return;      // no stream form
    const int tile = acquire_tile(sc.partials, &s_tile);
    if (tile >= num_tiles) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const long long p0 = static_cast<long long>(tile) * kPlanTile + threadIdx.x;
    int e[kPlanItems], a[kPlanItems], b[kPlanItems], tails[kPlanItems], tails_before[kPlanItems];
    bool more[kPlanItems];                              // the row has groups after this one
#pragma unroll
    for (int r = 0; r < kPlanItems; ++r) {
        const long long p = p0 + r * kPlanBlock;
        const int q = p < num_parts ? (place ? place[p] : static_cast<int>(p)) : -1;
        e[r] = q >= 0 && q < num_parts ? event_at[q] : -1;
        more[r] = p < num_parts && (info[p] & 2u) != 0;
    }
#pragma unroll
    for (int r = 0; r < kPlanItems; ++r) {
        const int2 x = e[r] >= 0 ? extent[e[r]] : make_int2(-1, 0);
        a[r] = x.x;
        b[r] = x.y;
    }
    unsigned partial = 0u, head = 0u;
    int ends_before[kPlanItems], rows_before[kPlanItems];
#pragma unroll
    for (int r = 0; r < kPlanItems; ++r) {
        const bool begins = a[r] >= 0;                  // the row's first piece
        tails[r] = e[r] >= 0 ? b[r] / kStreamWave - (a[r] & kStreamIdMask) / kStreamWave : 0;
        const bool part = e[r] >= 0 && (!begins || more[r] || tails[r] > 0);
        partial |= part ? 1u << r : 0u;
        head |= part && begins ? 1u << r : 0u;
        const uint64_t parts = __ballot(part), heads = __ballot(part && begins), rows = __ballot(begins);
        ends_before[r] = ballot_rank(parts);
        rows_before[r] = ballot_rank(heads);
        int incl = 0;
        if (__any(tails[r] > 0)) incl = wave_inclusive_scan(tails[r]);       // few waves see a piece that crosses
        tails_before[r] = incl - tails[r];
        if (lane == kWave - 1) {
            s_sum[0][r * kPlanWaves + wave] = (static_cast<uint64_t>(incl) << 31) + static_cast<uint64_t>(__popcll(parts));
            s_sum[1][r * kPlanWaves + wave] = (static_cast<uint64_t>(__popcll(rows)) << 31) + static_cast<uint64_t>(__popcll(heads));
        }
    }
    __syncthreads();
    if (wave < 2) {
        const uint64_t mine = s_sum[wave][lane];
        const uint64_t incl = wave_inclusive_scan_u64(mine);
        const uint64_t total = static_cast<uint64_t>(__shfl(static_cast<long long>(incl), kWave - 1, kWave));
        const uint64_t excl = tile_lookback(wave == 0 ? sc.ends_desc : sc.rows_desc, sc.partials, tile, total, mode);
        s_sum[wave][lane] = excl + incl - mine;
        if (tile == num_tiles - 1 && lane == 0) {
            const uint64_t all = excl + total;
            const int low = static_cast<int>(all & 0x7fffffffull), high = static_cast<int>(all >> 31);
            if (wave == 0) {
                sv.header->num_partials = low + high;
                *ends_total = low;
            } else {
                sv.header->num_fix = min(low, min(num_nodes, num_parts));
                sv.header->empty_rows = num_nodes - high;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPlanItems; ++r) {
        const long long p = p0 + r * kPlanBlock;
        if (p >= num_parts) continue;
        const bool part = (partial >> r) & 1u, begins = (head >> r) & 1u;
        int j = -1;
        if (part) {
            const uint64_t x = s_sum[0][r * kPlanWaves + wave], y = s_sum[1][r * kPlanWaves + wave];
            const int ea = ends_before[r] + static_cast<int>(x & 0x7fffffffull);
            const int ta = tails_before[r] + static_cast<int>(x >> 31);
            j = rows_before[r] + static_cast<int>(y & 0x7fffffffull) - (begins ? 0 : 1);
            if (begins && j < num_nodes && j < num_parts) {
                sv.frow[j] = rowp[p];
                sv.fptr[j] = ea + ta;
                ends0[j] = ea;
                tails0[j] = ta;
            }
            ends_at[p] = ea;
            tails_at[p] = ta;
        }
        fix_of[p] = j;
        if (place) event_of[p] = e[r];
    }
}

// The number of every partial sum into erow (a piece's end) and wtail (a chunk's tail); the header is completed.
__global__ __launch_bounds__(256) void plan_targets_kernel(StreamView sv, const int* __restrict__ event_of,
                                                          const int2* __restrict__ extent,
                                                          const int* __restrict__ fix_of, const int* __restrict__ ends_at,
                                                          const int* __restrict__ tails_at, const int* __restrict__ ends0,
                                                          const int* __restrict__ tails0, const int* __restrict__ ends_total,
                                                          int num_parts, int num_waves, PlanScans sc)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const bool error = sc.sort->error || sc.order->error || sc.partials->error;
    const bool usable = !error && sv.header->empty_groups == 0;
    if (p == 0) {
        sv.header->error = error ? 1 : 0;
        sv.header->valid = usable ? 1 : 0;
        if (usable) sv.fptr[sv.header->num_fix] = sv.header->num_partials;
    }
    if (!usable || p >= num_parts) return;
    const int j = fix_of[p];
    if (j < 0) return;
    const int e = event_of[p];
    sv.erow[e] = static_cast<int>(kStreamFlag) | (ends_at[p] + tails0[j]);
    const int2 x = extent[e];
    const int w0 = (x.x & kStreamIdMask) / kStreamWave, tails = x.y / kStreamWave - w0;
    if (tails > 0) {
        const int at = (j + 1 < sv.header->num_fix ? ends0[j + 1] : *ends_total) + tails_at[p];
        for (int k = 0; k < tails && w0 + k < num_waves; ++k) sv.wtail[w0 + k] = at + k;
    }
}

// ---------------------------------------------------------------- host
static size_t scan_state_bytes(long long n, int tile)
{
    const long long tiles = (n + tile - 1) / tile;
    return align256(sizeof(ScanState) + sizeof(uint64_t) * static_cast<size_t>(tiles > 0 ? tiles : 1));
}

static long long tiles_of(long long n, int tile) { return (n + tile - 1) / tile; }

// Workspace of a build: ten arrays of num_parts + 1 ints (some used twice, the later use in brackets), the sorted records, the
// adjacency bytes, the fill tiles' first entries, the radix histogram and its offsets, the scan states.
struct PlanTemp {
    int *keys_a, *keys_b, *order_a, *order_b, *rowp, *src, *ends_before, *event_at;
    int2* extent;                   // two slabs
    int4 *rec_in, *rec_out;         // rec_in = src, ends_before, extent (written after the sort)
    int *fix_of, *ends_at, *tails_at, *ends0, *tails0;      // = keys_a, keys_b, the spare order array, src, ends_before
    uint8_t* info;
    int *tile_q, *hist, *offsets, *ends_total;
    PlanScans scans;
    size_t bytes;
};
static PlanTemp plan_temp(char* base, long long num_parts, long long num_slots)
{
    PlanTemp t;
    size_t at = 0;
    auto take = [&](size_t bytes) { char* p = base + at; at += align256(bytes); return p; };
    const size_t slab = sizeof(int) * (static_cast<size_t>(num_parts) + 1);
    int** arrays[] = {&t.keys_a, &t.keys_b, &t.order_a, &t.order_b, &t.rowp, &t.src, &t.ends_before};
    for (int** a : arrays) *a = reinterpret_cast<int*>(take(slab));
    t.extent = reinterpret_cast<int2*>(take(2 * slab));
    t.event_at = reinterpret_cast<int*>(take(slab));
    t.info = reinterpret_cast<uint8_t*>(take(static_cast<size_t>(num_parts)));
    t.tile_q = reinterpret_cast<int*>(take(sizeof(int) * static_cast<size_t>(tiles_of(stream_padded_slots(num_slots), kFillTile) + 1)));
    const long long entries = tiles_of(num_parts, kSortTile) * kDigits;
    t.hist = reinterpret_cast<int*>(take(sizeof(int) * static_cast<size_t>(entries + 1)));
    t.offsets = reinterpret_cast<int*>(take(sizeof(int) * static_cast<size_t>(entries + 1)));
    auto state = [&](ScanState** st, uint64_t** desc, long long n, int tile) {
        char* p = take(scan_state_bytes(n, tile));
        *st = reinterpret_cast<ScanState*>(p);
        *desc = reinterpret_cast<uint64_t*>(p + sizeof(ScanState));
    };
    state(&t.scans.sort, &t.scans.sort_desc, entries, kScanTile);
    state(&t.scans.order, &t.scans.order_desc, num_parts, kPlanTile);
    state(&t.scans.partials, &t.scans.ends_desc, num_parts, kPlanTile);
    t.scans.rows_desc = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * static_cast<size_t>(tiles_of(num_parts, kPlanTile))));
    t.ends_total = reinterpret_cast<int*>(take(sizeof(int)));
    t.rec_in = reinterpret_cast<int4*>(t.src);                  // four slabs in a row
    t.rec_out = reinterpret_cast<int4*>(take(4 * slab));
    t.scans.order_tiles = static_cast<int>(tiles_of(num_parts, kPlanTile));
    t.scans.sort_tiles = 0;
    t.fix_of = t.keys_a; t.ends_at = t.keys_b; t.tails_at = nullptr; t.ends0 = t.src; t.tails0 = t.ends_before;
    t.bytes = at;
    return t;
}

size_t plan_workspace_bytes(long long num_parts, long long num_slots)
{
    if (num_parts <= 0) return 256;
    return plan_temp(nullptr, num_parts, num_slots).bytes;
}

// Where a build keeps the row of every group: a caller that already knows the rows leaves them there and passes the
// address as part2node.
int* plan_rows_in_workspace(void* workspace, long long num_parts, long long num_slots)
{
    return plan_temp(static_cast<char*>(workspace), num_parts, num_slots).rowp;
}

int workspace_pitch(int dim);   // aggregate.hip

static std::atomic<int> g_force_shift{0};     // process-wide knobs (tuning header), atomics like the ones below
// Plan policy.  Rows of up to 32 * keep slots are kept together instead of being cut at column-block borders, and
// single-group rows may be ordered by length class inside a block.  Negative = chosen per build from the kernel that
// will run over the plan:
//  * stream form (R-MAT 22, ms per epoch of aggregation): rows of up to 32 / 64 / 96 / 128 / 256 slots kept together
//    -> 4.11 / 4.04 / 4.05 / 4.08 / 4.08 without length classes, 4.15 with classes and 256.  Every gather instruction
//    is full whatever the lengths, so the classes only cost locality of the output rows (one-block plan of the
//    last-layer path: 0.227 -> 0.178 ms without them): keep 2, no classes.
//  * group kernel (runs over a plan when the shape is outside the stream kernel's: table of 4 GB or more, rows beyond
//    1024 bytes, stream mode off): equal gather steps per round matter, 256 slots with classes is its optimum and the
//    stream policy costs it 10 % (5.11 against 4.66 ms at R-MAT 22; 22.6 against 20.6 ms at R-MAT 24): keep 8, classes.
static std::atomic<int> g_keep_rows{-1};         // in units of 32 slots
static std::atomic<int> g_length_classes{-1};
void set_plan_length_classes(int on) { g_length_classes.store(on < 0 ? -1 : on ? 1 : 0); }
void set_plan_keep_rows(int keep) { g_keep_rows.store(keep < 0 ? -1 : keep); }
bool stream_covers(int num_nodes, int dim, int ld_in, const float* table);   // stream.hip
static void plan_policy(int num_nodes, int dim, int* keep_rows, int* length_classes)
{
    const bool stream = stream_covers(num_nodes, dim, workspace_pitch(dim), nullptr);
    const int keep = g_keep_rows.load(), classes = g_length_classes.load();
    *keep_rows = keep >= 0 ? keep : stream ? 2 : 8;
    *length_classes = classes >= 0 ? classes : stream ? 0 : 1;
}
void set_schedule_shift(int shift) { g_force_shift.store(shift); }

int schedule_shift(int dim)
{
    if (const int forced = g_force_shift.load(); forced > 0) return forced;
    // column blocks of at most 128K rows and 16 MB of feature rows.  Measured at R-MAT scale 22
    // (ms per epoch, 64- and 128-byte rows): 2^14 5.95, 2^15 5.74, 2^16 5.63, 2^17 5.60, 2^18 5.65,
    // 2^19 5.83 - the window all waves gather from has to stay resident in the memory-side cache,
    // not in one XCD's L2, and larger blocks leave fewer partial sums to combine
    const int row_bytes = 4 * workspace_pitch(dim);
    int shift = 17;
    while (shift > 8 && (static_cast<long long>(row_bytes) << shift) > (16ll << 20)) --shift;
    return shift;
}

// a later scan over the same state must not wipe the stall flag of an earlier one
__global__ void plan_scan_init_kernel(ScanState* st, uint64_t* desc, int num_tiles)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < num_tiles) desc[i] = kTileEmpty;
    if (i == 0) st->counter = 0;
}

// Every build gets a number of its own (> 0): it is written into the plan's header and remembered by the host with the
// header's counts, so that a kernel can tell the plan it was launched for from other bytes at the same address.
static std::atomic<int> g_plan_generation{0};
static int next_plan_generation()
{
    int g = g_plan_generation.fetch_add(1) + 1;
    if (g <= 0) { g_plan_generation.store(1); g = 1; }      // wrapped after 2^31 builds
    return g;
}
static int last_plan_generation() { return g_plan_generation.load(); }

// num_parts > 0
int check_plan_sizes(long long num_parts, long long num_slots, long long num_nodes, size_t plan_size, size_t workspace_bytes)
{
    if (plan_size < plan_bytes(num_parts, num_slots, num_nodes)) {
        set_error("build_plan: plan buffer smaller than eppgcn_plan_bytes(num_parts, num_slots, num_nodes)");
        return kErrInvalidArgument;
    }
    if (num_slots >= (1ll << 31) - kStreamWave) {            // the padded slots are counted in 32 bits too
        set_error("build_plan: slot count beyond 32-bit offsets");
        return kErrInvalidArgument;
    }
    if (plan_workspace_bytes(num_parts, num_slots) > workspace_bytes) {
        set_error("build_plan: workspace smaller than eppgcn_plan_workspace_bytes(num_parts, num_slots)");
        return kErrInvalidArgument;
    }
    return kOk;
}

int launch_build_plan(const int* part_ptr, const int* col, const int* part2node, const int* ids, int num_parts,
                      long long num_slots, int num_nodes, int shift, int dim, void* plan, size_t plan_size,
                      void* workspace, size_t workspace_bytes, const ScanState* upstream, hipStream_t stream)
{
    forget_stream_info(plan);
    int keep_rows, length_classes;
    plan_policy(num_nodes, dim, &keep_rows, &length_classes);
    if (num_parts <= 0) return kOk;
    if (int rc = check_plan_sizes(num_parts, num_slots, num_nodes, plan_size, workspace_bytes)) return rc;
    PlanTemp t = plan_temp(static_cast<char*>(workspace), num_parts, num_slots);
    const PlanView v = plan_view(plan, num_parts, num_nodes);
    const StreamView sv = stream_view(plan, num_parts, num_slots, num_nodes);
    const int slots = static_cast<int>(num_slots), padded = static_cast<int>(stream_padded_slots(num_slots));
    const int words = static_cast<int>(plan_single_words(num_nodes));

    // significant key bits; a plan in one block without length classes keeps the caller's order and needs no sort
    int bits = 0;
    while (bits < 30 && (static_cast<long long>(num_nodes > 0 ? num_nodes - 1 : 0) >> shift) >= (1ll << bits)) ++bits;
    if (length_classes) bits += 2;
    const int passes = (bits + 7) / 8;
    const int sort_tiles = static_cast<int>(tiles_of(num_parts, kSortTile));
    auto pass_bits = [&](int pass) { return bits - 8 * pass < 8 ? bits - 8 * pass : 8; };
    t.scans.sort_tiles = passes ? static_cast<int>(tiles_of(static_cast<long long>(sort_tiles) << pass_bits(0), kScanTile)) : 0;

    int init_blocks = (words + 255) / 256;
    if (init_blocks > 512) init_blocks = 512;
    if (init_blocks < 8) init_blocks = 8;
    hipLaunchKernelGGL(plan_init_kernel, dim3(init_blocks), dim3(256), 0, stream, sv.header, t.scans, v.single, sv.touched, words,
                       num_parts, slots, num_nodes, next_plan_generation(), upstream);
    EPPGCN_HIP(hipGetLastError());
    unsigned* keys_in = reinterpret_cast<unsigned*>(t.keys_a);
    unsigned* keys_out = reinterpret_cast<unsigned*>(t.keys_b);
    hipLaunchKernelGGL(plan_keys_kernel, dim3(sort_tiles), dim3(kKeysBlock), 0, stream, part_ptr, col, part2node, ids,
                       num_parts, num_nodes, shift > 31 ? 31 : shift, keep_rows * 32, length_classes,
                       passes ? 1 << pass_bits(0) : 1, sort_tiles, passes ? keys_in : nullptr, t.hist,
                       part2node == t.rowp ? nullptr : t.rowp, t.info, passes ? t.rec_in : nullptr, v.single, sv.touched, sv.header, t.scans.sort);
    EPPGCN_HIP(hipGetLastError());
    int* order = nullptr;            // after the last pass: the plan entry of every group
    int* spare = t.order_b;
    for (int pass = 0; pass < passes; ++pass) {
        const int nb = pass_bits(pass), digits = 1 << nb;
        const bool last_pass = pass + 1 == passes;
        const long long entries = static_cast<long long>(sort_tiles) * digits;
        const int scan_tiles = static_cast<int>(tiles_of(entries, kScanTile));
        if (pass > 0) {
            hipLaunchKernelGGL(plan_scan_init_kernel, dim3((scan_tiles + 255) / 256), dim3(256), 0, stream, t.scans.sort,
                               t.scans.sort_desc, scan_tiles);
            hipLaunchKernelGGL(radix_hist_kernel, dim3(sort_tiles), dim3(kSortBlock), 0, stream, keys_in, num_parts, 8 * pass,
                               digits, sort_tiles, t.hist);
            EPPGCN_HIP(hipGetLastError());
        }
        hipLaunchKernelGGL(exclusive_scan_kernel, dim3(scan_tiles), dim3(kScanBlock), 0, stream, t.hist, t.offsets,
                           static_cast<int>(entries), scan_tiles, t.scans.sort, t.scans.sort_desc, scan_mode());
        EPPGCN_HIP(hipGetLastError());
        int* out = order == t.order_a ? t.order_b : t.order_a;
        hipLaunchKernelGGL(radix_scatter_kernel, dim3(sort_tiles), dim3(kSortBlock), 0, stream, keys_in, order, keys_out, out,
                           num_parts, 8 * pass, nb, sort_tiles, t.offsets, t.rec_in, last_pass ? t.rec_out : nullptr);
        EPPGCN_HIP(hipGetLastError());
        unsigned* k = keys_in; keys_in = keys_out; keys_out = k;
        order = out;
        spare = out == t.order_a ? t.order_b : t.order_a;
    }
    t.tails_at = spare;
    hipLaunchKernelGGL(plan_order_kernel, dim3(t.scans.order_tiles), dim3(kPlanBlock), 0, stream, part_ptr,
                       passes ? t.rec_out : nullptr, t.rowp, t.info, num_parts, slots, t.scans.order_tiles, v, sv, t.src,
                       t.ends_before, t.extent, t.event_at, t.tile_q, t.scans.order, t.scans.order_desc, scan_mode(),
                       t.scans.sort);
    EPPGCN_HIP(hipGetLastError());
    int* event_of = passes ? reinterpret_cast<int*>(t.rec_out) : t.event_at;       // the records have been read
    if (padded > 0) {
        const int fill_tiles = static_cast<int>(tiles_of(padded, kFillTile));
        hipLaunchKernelGGL(plan_fill_kernel, dim3(fill_tiles), dim3(256), 0, stream, col, v, sv, t.src, t.ends_before, t.tile_q,
                           num_parts, slots, padded, num_nodes, fill_tiles, t.scans);
        EPPGCN_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(plan_partials_kernel, dim3(t.scans.order_tiles), dim3(kPlanBlock), 0, stream, t.rowp, t.info, order, t.event_at,
                       event_of, t.extent, num_parts, num_nodes, t.scans.order_tiles, sv, t.fix_of, t.ends_at, t.tails_at,
                       t.ends0, t.tails0, t.ends_total, t.scans, scan_mode());
    EPPGCN_HIP(hipGetLastError());
    hipLaunchKernelGGL(plan_targets_kernel, dim3((num_parts + 255) / 256), dim3(256), 0, stream, sv, event_of, t.extent,
                       t.fix_of, t.ends_at, t.tails_at, t.ends0, t.tails0, t.ends_total, num_parts, padded / kStreamWave, t.scans);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

// ---------------------------------------------------------------- what the host knows about built plans
}  // namespace eppgcn

#include <map>
#include <mutex>

namespace eppgcn {

static std::mutex g_info_mutex;
static std::map<const void*, StreamInfo> g_infos;

const StreamInfo* find_stream_info(const void* plan, StreamInfo* copy)
{
    std::lock_guard<std::mutex> lock(g_info_mutex);
    auto it = g_infos.find(plan);
    if (it == g_infos.end()) return nullptr;
    *copy = it->second;
    return copy;
}
void forget_stream_info(const void* plan)
{
    std::lock_guard<std::mutex> lock(g_info_mutex);
    g_infos.erase(plan);
}
void remember_stream_info(const void* plan, const StreamInfo& info)
{
    std::lock_guard<std::mutex> lock(g_info_mutex);
    g_infos[plan] = info;
}

// Synchronises the stream and reports (once) a header mismatch that a stream or fix-up kernel has seen on the current
// device since the last report.
int read_aggregation_status(hipStream_t stream)
{
    int* words = nullptr;
    if (int rc = plan_fault_address(&words)) return rc;
    int host[kPlanFaultWords] = {0, 0, 0, 0};
    EPPGCN_HIP(hipMemcpyAsync(host, words, sizeof(host), hipMemcpyDeviceToHost, stream));
    EPPGCN_HIP(hipStreamSynchronize(stream));
    if (!host[0]) return kOk;
    if (int rc = launch_zero_words(words, kPlanFaultWords, stream)) return rc;
    set_error(std::string("an aggregation call was given a plan whose header in memory is not the one the library read at "
                          "that address (seen by the ") + (host[1] == 2 ? "fix-up" : "stream") + " kernel: build " +
              std::to_string(host[2]) + " expected, " + std::to_string(host[3]) +
              " found); that call wrote no output.  The plan's memory was overwritten or replaced: rebuild the plan, or "
              "call eppgcn_plan_release when a plan's memory is given up");
    return kErrPlanMismatch;
}

const void* plan_header_address(const void* plan, long long num_parts, long long num_slots, long long num_nodes)
{
    return stream_view(const_cast<void*>(plan), num_parts, num_slots, num_nodes).header;
}

// Records the plan's header, which is read from the device with a wait for the stream unless the caller has a copy of it
// (`read`, complete); the return code tells whether a look-back scan of the build stalled.
int read_plan_status(const void* plan, long long num_parts, long long num_slots, long long num_nodes,
                     long long* partial_rows, const void* read, hipStream_t stream)
{
    if (partial_rows) *partial_rows = 0;
    if (num_parts <= 0) return kOk;
    StreamInfo info;
    info.num_parts = num_parts; info.num_slots = num_slots; info.num_nodes = num_nodes;
    if (read) {
        memcpy(&info.header, read, sizeof(StreamHeader));
    } else {
        EPPGCN_HIP(hipMemcpyAsync(&info.header, plan_header_address(plan, num_parts, num_slots, num_nodes), sizeof(StreamHeader),
                                  hipMemcpyDeviceToHost, stream));
        EPPGCN_HIP(hipStreamSynchronize(stream));
    }
    {   // the address of the mismatch mark on this device is looked up here, outside any graph capture
        int* words = nullptr;
        if (int rc = plan_fault_address(&words)) return rc;
    }
    // only a header that a build of this process wrote for these sizes is taken on: its counts size the launches
    const StreamHeader& h = info.header;
    const long long waves = stream_padded_slots(num_slots) / kStreamWave;
    const bool plausible = h.magic == kPlanMagic && h.generation > 0 && h.generation <= last_plan_generation() &&
                           h.num_parts == num_parts && h.num_nodes == num_nodes && h.num_slots == num_slots &&
                           h.num_events >= 0 && h.num_events <= num_parts && h.num_partials >= 0 &&
                           h.num_partials <= num_parts + waves && h.num_fix >= 0 && h.num_fix <= num_nodes &&
                           h.num_fix <= h.num_partials && h.empty_rows >= 0 && h.empty_rows <= num_nodes;
    if (!plausible) {
        forget_stream_info(plan);
        set_error("plan_status: the memory at `plan` does not hold a plan built with these sizes (no build has "
                  "finished there, or its bytes were overwritten); rebuild it with eppgcn_build_plan");
        return kErrPlanMismatch;
    }
    if (info.header.error) {
        forget_stream_info(plan);
        set_error("look-back scan stalled: a tile waited past its spin limit, or the split before the plan found other counts "
                  "than it was given; the plan is invalid");
        return kErrScanStalled;
    }
    remember_stream_info(plan, info);
    if (partial_rows && info.header.valid) *partial_rows = info.header.num_partials;
    return kOk;
}

}  // namespace eppgcn

// Routing layout: per-expert histograms, device-wide scan, stable token-order slots, slot-order list.

#include <ctime>

#include <mutex>

#include "nanoep_ahead.h"
#include "nanoep_device.h"

// Device memory of nanoep_layout_static: the layout kernels' workspace (histogram
// rows) for callers that cannot allocate.  Every GPU holds its own copy of the array
// at its own address until the process ends; host code only ever uses the address that
// hipGetSymbolAddress returns for the current device, never the array's name.
static __device__ __align__(256) unsigned char scratch[NANOEP_STATIC_SCRATCH_BYTES];

namespace nanoep {
namespace {

// What the launch plans below depend on besides the batch: the forced settings and the device's XCD
// count and L2 size (the rows of one window should fit an XCD's L2, since the dispatch walks the
// slot-order list window by window and wants every re-use of a source row to hit that cache).
struct Knobs {
    int window_tokens;
    int layout_launches;
    int cus;
    int xcds;
    int64_t l2_bytes;
};

Knobs current_knobs() {
    const Tuning tuning = current_tuning();
    const Topology topology = current_topology(tuning);
    return {tuning.window_tokens, tuning.layout_launches, topology.cus, topology.xcds, topology.l2_bytes};
}

// The slot-order buffer holds T rounded up to this many tokens' choices.
constexpr int kOrderTokens = 256;
// Largest window: the run of consecutive tokens the slot-order list is ordered by.
constexpr int kMaxWindowTokens = 1024;
// Largest batch that takes windows of more than 256 tokens.
constexpr int64_t kMaxWideWindowBatch = int64_t{1} << 18;
// Most threads of a layout workgroup.
constexpr int kLayoutThreads = 1024;
constexpr int kLayoutWaves = kLayoutThreads / kWave;
// Most tokens of an assignment workgroup (four words of the bit matrix) and the (token, choice) pairs it aims at.
constexpr int kMaxBlockTokens = 128;
constexpr int kBlockPairs = 512;
// Chunks of pairs a wavefront fetches at a time where it counts more than one.
constexpr int kChunks = 4;
// Chunks of its block an assignment wavefront takes: one, so that a workgroup is done soon, until the launch has more
// wavefronts than half the device holds.  From there on it is the rounds of workgroups that cost, each the whole chain of round
// trips, and fewer wavefronts with more chunks are fewer rounds: two behind histogram rows, where a workgroup's
// wavefronts also share the summing of the rows, four behind a scan.  Launch period of the layout, one chunk -> two (four):
// 32768 x 16, 64 experts 17.8 -> 15.0 (15.4) us, 65536 x 8, 64 18.5 -> 15.7 (15.9), 65536 x 32, 256 89 -> 70 (71), 131072 x 8, 64
// 31 -> 25.5 (25.8); behind a scan 400000 x 8, 64 129 -> 97 (96), 400000 x 10, 64 139 -> 117 (107).
constexpr int kSummedChunks = 2;
constexpr int kScannedChunks = 4;
constexpr int64_t kOneChunkWaves = 4096;
// Pairs up to which every workgroup counts the whole batch by itself.  One launch against two, launch period:
// 512 x 8, 128 experts 5.1 against 7.5 us, 2048 x 2, 8 experts 5.8 against 7.5, 1537 x 4, 60 experts 6.0
// against 7.7, 1024 x 8, 128 experts 7.2 against 7.5, and 8.3 against 7.5 us at 4096 x 2 with 8 experts, where
// the LDS additions meet on few words.
constexpr int64_t kDirectPairs = 7168;
// Histogram rows: the most every assignment workgroup sums by itself (a scan launch between, launch period:
// 131072 tokens x 8, 256 experts, 512 rows 69 against 114 us; 262144 x 4, 64 experts, 1024 rows 58 against 64;
// 524288 x 8, 2048 rows 251 against 161), and how many a wavefront fetches at a time (their number is padded
// to a multiple of it).
constexpr int64_t kSummedHistograms = 1024;
constexpr int kSumRows = 16;

// Tokens of one window of the slot-order list.
//  * `hidden` (bf16 elements of a payload row, 0 = not known) sizes the window so that its rows fit an
//    XCD's L2 with a sixteenth to spare for the write stream (a window that fills the L2 to the
//    brim loses what the prefetch brought in: 4096 x 4096 top-2 18.9 -> 18.3 us cold, 14.9 -> 12.8 us
//    cache resident with half the window): 512 tokens up to 3840 elements, 256 up to 7680 (and when
//    it is not known), then 128, 64.
//    Rows of up to 1024 elements take 1024 tokens (half the L2: at 2048 elements a 1024-token window
//    measured 8 % slower than a 512-token one, at 1024 and 512 elements 5 and 7 % faster).
//  * The dispatch hands every XCD whole windows when there are at least as many as XCDs (twice as
//    many for 1024-token windows): batches of more than 256 tokens take smaller windows (down to 64
//    tokens) to get there.
// (sizes above are those of a 4 MiB L2 and 8 XCDs)
int layout_window_tokens(int64_t tokens_total, int hidden, const Knobs& knobs) {
    // WINDOW_TOKENS forces a window: any multiple of 32 up to 256, or 512 / 1024
    const int forced = knobs.window_tokens;
    if (forced >= 32 && forced % 32 == 0 && (forced <= 256 || forced == 512 || forced == 1024) && tokens_total > 256)
        return forced;
    int window = 256;
    if (hidden > 0)
        for (window = kMaxWindowTokens;
             window > 64 && static_cast<int64_t>(window) * hidden * 2 > (window > 512 ? knobs.l2_bytes / 2 : knobs.l2_bytes - knobs.l2_bytes / 16);
             window /= 2) {
        }
    if ((tokens_total <= 256 || tokens_total > kMaxWideWindowBatch) && window > 256)
        window = 256;
    while (tokens_total > 256 && window > 64 && (tokens_total + window - 1) / window < (window > 512 ? 2 * knobs.xcds : knobs.xcds))
        window /= 2;
    return window;
}

// LDS of a workgroup: three counters an expert (and one row more for received tokens), then a bit
// matrix of one bit a token.
size_t layout_lds(int64_t local_experts, int64_t bit_words) {
    return static_cast<size_t>(local_experts + 1) * 12 + static_cast<size_t>(local_experts) * bit_words * 4 + 16;
}

bool layout_supports(int64_t local_experts) { return local_experts > 0 && (local_experts + 1) * 16 <= static_cast<int64_t>(kLayoutLdsBudget); }

// Tokens of one assignment workgroup: whole words of the bit matrix, a whole number of workgroups a window,
// a chunk a wavefront; more once that makes two workgroups a compute unit.
int layout_block_tokens_of(int64_t tokens_total, int window, int topk, int64_t local_experts) {
    for (int tokens = kMaxBlockTokens; tokens > 32; tokens -= 32)
        if (window % tokens == 0 && tokens * topk <= (tokens_total > 256 * (kBlockPairs / topk) ? 2 : 1) * kBlockPairs &&
            layout_lds(local_experts, tokens / 32) <= kLayoutLdsBudget)
            return tokens;
    return 32;
}

// Tokens of a histogram row: at least 64 where the window allows it, and more while an assignment wavefront
// has more batches of rows to fetch than batches of ids between the start of its block's row and the block.
int layout_histogram_tokens(int64_t tokens_total, int window, int block_tokens, int topk, int64_t local_experts) {
    int tokens = block_tokens < 64 && window % 64 == 0 ? 64 : block_tokens;
    while (window % (2 * tokens) == 0) {
        const int64_t rows = (tokens_total + tokens - 1) / tokens;
        const int64_t row_tasks = (rows + kSumRows - 1) / kSumRows * ((local_experts + kWave - 1) / kWave);
        const int64_t id_batches = static_cast<int64_t>(2 * tokens - block_tokens) * topk / (kWave * kChunks);
        if (row_tasks <= 8 || row_tasks <= id_batches)
            break;
        tokens *= 2;
    }
    return tokens;
}

// Source rows that a layout which knows of them reads ahead for the dispatch behind it (read_source_ahead): up to 4 MiB beside the
// assignment while that launch then has a workgroup for no more than three quarters of the compute units, up to 2 MiB until it has one for
// each, nothing beyond (what waits for a place holds the launch up); up to 8 MiB beside the histogram rows of batches of 2^18 pairs and more,
// whose assignment never has the room.  Both launches wait for round trips, not for bytes, until the reads go on longer than they do.
// Layout and dispatch, launch period, no row used again within 768 MiB (one x, in the caches), nothing -> this rule:
// 4 MiB: 800 x 7168 top-8 25.0 -> 24.1 us (21.9 -> 22.0), 1024 x 2048 top-4 11.6 -> 10.4 (10.6 -> 10.6), 1537 x 2816 top-6 22.9 -> 21.4
// (17.9 -> 17.9), 2048 x 5120 top-8 34.4 -> 34.0 (31.6 -> 31.6), 3000 x 4096 43.9 -> 43.0 (38.5 -> 38.3), 4096 x 4096 top-2 25.4 -> 25.2 (20.4 ->
// 20.2), 4096 x 7168 top-8 86.0 -> 86.0 (82.1 -> 81.7), 6000 x 2048 49.5 -> 48.2 (43.1 -> 42.9), 12000 x 4096 top-2 59.2 -> 58.7 (55.1 -> 54.3);
// 2 MiB: 8192 x 2048 top-8 62.1 -> 61.6 (level), 16384 x 4096 top-2 75.9 -> 75.5 (64.8 -> 64.5), 28000 x 512 top-8 54.7 -> 54.5 (48.1 -> 47.9); with
// 4 MiB there 8192 x 4096 top-2 44.5 -> 45.0, 16384 x 4096 top-2 76.9, 16384 x 2048 top-4 67.2 -> 67.4; with 4 MiB beside 235 to 251 workgroups
// 30000 x 512 58.9 -> 60.9 (49.7 -> 50.4), 32000 x 512 62.2 -> 65.3 (55.3 -> 56.1), 16000 x 1024 59.3 -> 60.3 (51.9 -> 52.2).
// The device's compute units count also where a stream's mask (a compute-unit budget) leaves fewer: the workgroups that wait there hold up a layout
// that is a smaller part of the pass.  32 of 256: 256 x 4096 top-8 24.1 -> 23.1 (18.6 -> 18.7), 800 x 7168 105.5 -> 103.7 (91.1 -> 92.1), 1537 x 2816
// 73.7 -> 69.2 (55.6 -> 55.8), 4096 x 4096 top-2 75.3 -> 74.6 (63.9 -> 64.1), 4096 x 7168, 8192 x 2048 and 8192 x 4096 top-2 level; 64: 1537 x 2816 46.3
// -> 42.8, 4096 x 4096 top-2 45.2 -> 45.5 (38.4 -> 38.5); 128: 1537 x 2816 32.4 -> 29.7, 8192 x 2048 84.2 -> 84.4 (78.4 -> 78.5).
// 8 MiB, no row used again within 768 MiB it is level, one x in the caches it gains: 2^18 pairs 32768 x 512 top-8 61.3 -> 61.2 (55.4 -> 54.6), 32768 x
// 1024 106.7 -> 106.7 (96.5 -> 95.4), 32768 x 2048 202.3 -> 201.3 (179.8 -> 178.6), 65536 x 512 top-4 77.7 -> 77.9 (63.7 -> 63.1); more: 44000 x
// 1024 top-6 121.9 -> 121.0 (106.2 -> 105.4), 40000 x 1024 top-8 130.9 -> 131.4 (121.6 -> 120.6), 65536 x 512 114.4 -> 113.7 (101.5 -> 101.2), 65536 x 1024
// 198.1 -> 197.2 (178.4 -> 178.3), 131072 x 256 143.5 -> 141.8 (118.2 -> 118.5).  At 2^17 pairs it is a trade: 16384 x 1024 top-8 55.9 -> 56.2
// (51.1 -> 50.8), 16384 x 4096 191.6 -> 192.4 (169.8 -> 169.1), 32768 x 1024 top-4 68.2 -> 69.3 (59.1 -> 58.3).  From about 160000 pairs on it would
// gain already where the assignment has no room (31000 x 512 top-8 59.4 -> 58.8 (51.7 -> 50.5), 48000 x 512 top-4 58.0 -> 58.0 (49.9 -> 48.8)).
constexpr int64_t kHistogramAheadPairs = int64_t{1} << 18;
constexpr int64_t kHistogramAheadBytes = int64_t{8} << 20;
constexpr int64_t kAssignAheadBytes = int64_t{4} << 20;

// What a histogram row holds besides its counts.
struct RowInfo {
    uint32_t received;  // tokens with any valid choice
    uint32_t assigned;  // valid choices
    int32_t status;     // routing status bits
    uint32_t unused;
};

struct LayoutWorkspace {
    int32_t* histograms;  // [rows][L]
    RowInfo* rows;        // [rows]
    int64_t* totals;      // [1] total assignments, handed from the scan kernel to the assignment kernel
    size_t bytes;
};

int64_t padded_rows(int64_t rows) { return (rows + kSumRows - 1) / kSumRows * kSumRows; }

// Sized for the most histogram rows a payload of any width can lead to, one every 64 tokens (32 under a
// forced window that is no multiple of 64), padded.  The total has always had room for a word a (token, choice)
// pair and a token as well, and callers hold buffers and one fixed array of that size: it stays.
LayoutWorkspace carve_layout_workspace(void* base, int64_t tokens, int topk, int64_t local_experts, const Knobs& knobs) {
    const int row_tokens = knobs.window_tokens % 64 == 0 ? 64 : 32;
    const int64_t rows = !layout_supports(local_experts) ? 0 : padded_rows((tokens + row_tokens - 1) / row_tokens);
    auto* cursor = static_cast<uint8_t*>(base);
    size_t offset = 0;
    LayoutWorkspace ws{};
    ws.histograms = reinterpret_cast<int32_t*>(cursor + offset);
    offset = align_up(offset + static_cast<size_t>(rows) * (local_experts + 1) * 4, 256);
    ws.rows = reinterpret_cast<RowInfo*>(cursor + offset);
    offset = align_up(offset + static_cast<size_t>(rows) * sizeof(RowInfo), 256);
    ws.totals = reinterpret_cast<int64_t*>(cursor + offset);
    offset = align_up(offset + static_cast<size_t>(tokens) * topk * 4, 256);
    offset = align_up(offset + static_cast<size_t>(tokens) * 4, 256);
    offset = align_up(offset + 8, 256);
    ws.bytes = offset + 256;
    return ws;
}

struct LayoutArgs {
    const int64_t* topk_idx;  // [T][K]
    int32_t* histograms;      // [rows][L]
    RowInfo* rows;
    uint32_t tokens;
    uint32_t topk;
    uint32_t experts;
    uint32_t chunk_tokens;  // whole tokens a wavefront covers at a time: 64 / K
    uint32_t chunk_pairs;   // chunk_tokens * K
    uint32_t topk_magic;    // lane / K = (lane * topk_magic) >> 16
    uint32_t waves;         // of a workgroup
    uint32_t block_tokens;  // tokens of an assignment workgroup
    uint32_t row_tokens;    // tokens of a histogram row: a multiple of block_tokens, a divisor of window_tokens
    uint32_t row_magic;     // fast divisor by row_tokens
    uint32_t row_shift;
    uint32_t window_tokens;  // of the slot-order list, a multiple of block_tokens
    uint32_t window_magic;   // fast divisor by window_tokens
    uint32_t window_shift;
    uint32_t row_count;    // histogram rows
    uint32_t row_batches;  // ... in batches of kSumRows (the rows that pad the last one are zero)
    uint32_t strips;       // experts in units of 64
    uint32_t strips_magic;  // fast divisor by it
    uint32_t strips_shift;
    uint32_t per_thread;    // experts a thread takes in the scans
    uint32_t expert_waves;  // wavefronts that have any
    uint32_t check_tokens;  // tokens of a row whose bits fit the histogram kernel's LDS at a time
    uint32_t expand;
    uint32_t alignment_magic;  // fast divisor by the alignment
    uint32_t alignment_shift;
    int64_t alignment;
    int64_t* totals;
    int64_t* expert_counts;
    int64_t* expert_offsets;
    int64_t* send_counts;
    int64_t* recv_rank_prefix;
    int64_t* host_counts;
    int64_t* snapshot;
    int32_t* recv_metadata;
    int64_t* dst_slots;
    int32_t* token_slots;  // or null
    int64_t* slot_order;   // or null
    uint64_t list_entries;  // of the slot-order buffer, without its count word
    uint32_t blocks;
};

// Workgroups behind a layout launch's own: they read the rows that the dispatch of this batch starts with.  Workgroup b (on
// XCD b % count) reads on from the start of that XCD's share of the rows.  A batch of at least as many windows as XCDs is given
// to them in contiguous shares, so an XCD's L2 then holds the first rows of its first window before the dispatch is launched, and the
// last-level cache what does not fit.  Of fewer windows, or of the one of up to 256 tokens, every XCD copies rows from all of the batch:
// those find them in the last-level cache.  (The walk's own prefetch is off for a batch of one window, where it stands in front of
// one XCD's copies; these reads are ahead of all copies.)  Layout and dispatch, launch period, no row used again within 768 MiB, nothing ->
// read ahead: 128 x 7168 top-8 10.4 -> 9.6 us, 200 x 5120 top-6 10.3 -> 9.8, 256 x 4096 10.5 -> 9.7, 256 x 7168 13.2 -> 12.8, top-2 9.6 -> 9.4;
// with one x, in the caches, all within 0.1.  Nothing depends on these reads.
struct SourceAhead {
    const u32x4* x;        // [T][row vectors], or null
    uint32_t work_blocks;  // workgroups of the launch's own
    uint32_t vectors;      // of all source rows
    uint32_t share;        // of an XCD's part of them
    XcdMap xcds;
};

__device__ __forceinline__ void read_source_ahead(const SourceAhead& s, uint32_t waves) {
    const uint32_t ordinal = fast_divide(blockIdx.x - s.work_blocks, s.xcds.magic, s.xcds.shift);
    const uint32_t xcd = blockIdx.x - fast_divide(blockIdx.x, s.xcds.magic, s.xcds.shift) * s.xcds.count;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const AheadRange range = ahead_range(s.vectors, s.share, xcd, ordinal, waves, wave);
    if (range.first >= range.end)
        return;
    u32x4 fetched[kAheadLoads];
#pragma unroll
    for (int u = 0; u < kAheadLoads; ++u)
        fetched[u] = s.x[ahead_vector(range, u, threadIdx.x % kWave)];
#pragma unroll
    for (int u = 0; u < kAheadLoads; ++u)
        asm volatile("" ::"v"(fetched[u].x), "v"(fetched[u].y), "v"(fetched[u].z), "v"(fetched[u].w));
}

// Where an assignment workgroup gets the counts of the other workgroups' tokens from.
enum LayoutSource {
    kDirect,   // it counts all of the batch's ids itself: one launch, nothing passes through memory
    kSummed,   // from the histogram rows layout_histogram_kernel left, which it sums itself
    kScanned,  // from the prefixes layout_scan_kernel made of those rows
};

__device__ __forceinline__ int64_t round_up_to(int64_t count, const LayoutArgs& a) {
    if (a.alignment == 1 || count == 0)
        return count;
    return static_cast<int64_t>(fast_divide(static_cast<uint32_t>(count) - 1u, a.alignment_magic, a.alignment_shift) + 1u) * a.alignment;
}

// Wavefronts take (token, choice) pairs in chunks of whole tokens: pair token * K + k of the chunk on
// that lane, the lanes left over idle.  A chunk's pairs are consecutive in every [T][K] array, so their
// addresses are a uniform base plus the lane.  These kernels run a handful of workgroups and last a few
// microseconds: what they cost is the instructions of a workgroup's wavefronts one after the other on
// its compute unit (a vector instruction of 16 wavefronts is 7 ns) and the round trips between them.
struct PairLane {
    uint32_t lane;
    uint32_t token;    // of the chunk
    uint32_t k;
    uint64_t earlier;  // the lanes of the same token's earlier choices
};

__device__ __forceinline__ PairLane pair_lane(const LayoutArgs& a) {
    PairLane at;
    at.lane = threadIdx.x % kWave;
    at.token = (at.lane * a.topk_magic) >> 16;
    at.k = at.lane - at.token * a.topk;
    at.earlier = ((uint64_t{1} << at.k) - 1u) << (at.lane - at.k);
    return at;
}

// Pairs of the chunk that starts at token `first` of a range that ends at `end`.
__device__ __forceinline__ uint32_t pairs_of_chunk(const LayoutArgs& a, uint32_t first, uint32_t end) {
    if (first >= end)
        return 0;
    return end - first < a.chunk_tokens ? (end - first) * a.topk : a.chunk_pairs;
}

// The lane's id of that chunk, -1 when it has none.
__device__ __forceinline__ int64_t fetch_id(const LayoutArgs& a, const PairLane& at, uint32_t first, uint32_t end) {
    int64_t id = -1;
    if (at.lane < pairs_of_chunk(a, first, end))
        id = (a.topk_idx + static_cast<uint64_t>(first) * a.topk)[at.lane];
    return id;
}

__device__ __forceinline__ bool names_expert(int64_t id, const LayoutArgs& a) { return static_cast<uint64_t>(id) < static_cast<uint64_t>(a.experts); }

// (the layout goes on with what it takes for masked choices, and stays inside its bounds)
__device__ __forceinline__ int check_id(int64_t id, const LayoutArgs& a) { return id == -1 || names_expert(id, a) ? 0 : NANOEP_ROUTING_BAD_EXPERT; }

// Sets the token's bit in its expert's row of the bit matrix; true when it was set before (another
// choice of the token names the same expert).
__device__ __forceinline__ bool set_token_bit(uint32_t* bits, uint32_t words, int64_t id, uint32_t token) {
    const uint32_t bit = 1u << (token % 32);
    return (atomicOr(&bits[static_cast<uint32_t>(id) * words + token / 32], bit) & bit) != 0;
}

// Number of tokens of a chunk that open with this lane's pair: the token's first valid choice.
__device__ __forceinline__ uint32_t count_opening(uint64_t valid_mask, bool counted, const PairLane& at) {
    return __popcll(__ballot(counted && (valid_mask & at.earlier) == 0));
}

// The routing status bits any lane of the wavefront has.
__device__ __forceinline__ int wave_status(int bad) {
    return (__ballot(bad & NANOEP_ROUTING_BAD_EXPERT) ? NANOEP_ROUTING_BAD_EXPERT : 0) | (__ballot(bad & NANOEP_ROUTING_DUPLICATE) ? NANOEP_ROUTING_DUPLICATE : 0);
}

// Zeroes `words` words of LDS (16-byte aligned, room up to the next multiple of four).
__device__ __forceinline__ void clear_lds(uint32_t* lds, uint32_t words, uint32_t threads) {
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (uint32_t i = threadIdx.x; i < (words + 3) / 4; i += threads)
        reinterpret_cast<u32x4*>(lds)[i] = zero;
}

// Names a word of every cache line of the arguments: they arrive with the first batch of scalar loads, and what is
// asked for later is in the scalar cache.  Left where it is first used, a line is a round trip to memory of its own on the
// way of every wavefront.  Launch period, without -> with: one launch 256 x 8, 64 experts 4.51 -> 4.37 us, 1537 x 4, 60 experts 6.28 -> 6.13; two
// launches 1537 x 6 7.90 -> 7.54, 4096 x 8, 64 experts 8.01 -> 7.61, 8192 x 8, 128 experts 9.08 -> 8.67, 32768 x 8 12.5 -> 12.1.  (Barriers that
// wait for LDS alone, in place of __syncthreads(), give nothing: 0.00 +- 0.05 us over the same batches.)
__device__ __forceinline__ void fetch_layout_arguments(const LayoutArgs& a) {
    static_assert(sizeof(LayoutArgs) <= 4 * 64, "one word of every line");
    NANOEP_FETCH_ARGS_4(a.topk_idx, a.per_thread, a.alignment, a.dst_slots);
    NANOEP_FETCH_ARGS_2(a.blocks, a.blocks);
}

// One histogram row: the experts' counts among `row_tokens` tokens, and their RowInfo.  Rows behind the
// batch's end come out zero.
__global__ void __launch_bounds__(kLayoutThreads) layout_histogram_kernel(const LayoutArgs a, const uint32_t waves, const SourceAhead ahead) {
    extern __shared__ __align__(16) uint32_t histogram_lds[];
    __shared__ RowInfo info;
    NANOEP_FETCH_ARGS_4(a.topk_idx, a.experts, a.check_tokens, waves);
    NANOEP_FETCH_ARGS_2(ahead.x, ahead.work_blocks);
    if (blockIdx.x >= ahead.work_blocks) {
        read_source_ahead(ahead, waves);
        return;
    }
    const uint32_t words = a.check_tokens / 32;
    const uint32_t counter_words = (a.experts + 3) / 4 * 4;
    uint32_t* counts = histogram_lds;                // [L]
    uint32_t* bits = histogram_lds + counter_words;  // [L][words]: check_tokens of the row at a time
    const PairLane at = pair_lane(a);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t step = waves * a.chunk_tokens;
    const uint32_t first = blockIdx.x * a.row_tokens;
    const uint32_t row_end = first + a.row_tokens < a.tokens ? first + a.row_tokens : a.tokens;
    int bad = 0;
    uint32_t received = 0, assigned = 0;
    uint32_t set_first = first;
    do {
        const uint32_t end = set_first + a.check_tokens < row_end ? set_first + a.check_tokens : row_end;
        uint32_t chunk = set_first + wave * a.chunk_tokens;
        int64_t id[kChunks];
#pragma unroll
        for (int j = 0; j < kChunks; ++j)
            id[j] = fetch_id(a, at, chunk + j * step, end);
        if (set_first == first) {
            clear_lds(histogram_lds, counter_words + a.experts * words, waves * kWave);
            if (threadIdx.x == 0)
                info = RowInfo{0, 0, 0, 0};
        } else {
            __syncthreads();
            clear_lds(bits, a.experts * words, waves * kWave);
        }
        __syncthreads();
        while (chunk < end) {
#pragma unroll
            for (int j = 0; j < kChunks; ++j) {
                const uint32_t chunk_first = chunk + j * step;
                if (chunk_first >= end)
                    break;  // (the same for the whole wavefront)
                const bool valid = names_expert(id[j], a);
                const uint64_t valid_mask = __ballot(valid);
                if (valid) {
                    atomicAdd(&counts[static_cast<uint32_t>(id[j])], 1u);
                    if (set_token_bit(bits, words, id[j], chunk_first - set_first + at.token))
                        bad |= NANOEP_ROUTING_DUPLICATE;
                }
                bad |= check_id(id[j], a);
                received += count_opening(valid_mask, valid, at);
                assigned += __popcll(valid_mask);
            }
            chunk += kChunks * step;
            if (chunk < end) {
#pragma unroll
                for (int j = 0; j < kChunks; ++j)
                    id[j] = fetch_id(a, at, chunk + j * step, end);
            }
        }
        set_first += a.check_tokens;
    } while (set_first < row_end);
    bad = wave_status(bad);
    if (at.lane == 0 && (assigned != 0 || bad != 0)) {
        atomicAdd(&info.received, received);
        atomicAdd(&info.assigned, assigned);
        atomicOr(&info.status, bad);
    }
    __syncthreads();
    int32_t* row = a.histograms + static_cast<uint64_t>(blockIdx.x) * a.experts;
    for (uint32_t i = threadIdx.x; i < a.experts; i += waves * kWave)
        row[i] = static_cast<int32_t>(counts[i]);
    if (threadIdx.x == 0)
        a.rows[blockIdx.x] = info;
}

// The mailbox: words 1 to 3, and word 0 once they have arrived.  The stores are system-scope writes to
// host memory and the wait between them is all the order they need: nothing else is published with
// them, so no cache is written back (a release fence here writes back the XCD's L2, every token's part
// of the handle included).
__device__ __forceinline__ void publish_counts(int64_t* host_counts, int64_t received, int64_t capacity, int64_t assigned, int64_t status) {
    __hip_atomic_store(&host_counts[1], capacity, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&host_counts[2], assigned, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&host_counts[3], status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(&host_counts[0], received, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Single workgroup.  Phase 1 turns every column of the histogram rows into its exclusive prefix
// (threads are spread over columns x row segments so small expert counts still use the whole
// workgroup).  Phase 2 scans the aligned expert totals.
__global__ void __launch_bounds__(kScanThreads) layout_scan_kernel(const LayoutArgs a) {
    extern __shared__ int32_t column_total[];  // [L+1]; column L is the received tokens
    __shared__ int32_t partial[kScanThreads];
    __shared__ int64_t scan[kScanThreads];
    __shared__ int64_t assignments[kScanThreads];
    __shared__ int status_bits;

    const int tid = threadIdx.x;
    const int experts = static_cast<int>(a.experts);
    const int rows = experts + 1;
    const int num_blocks = static_cast<int>(a.row_count);
    if (tid == 0)
        status_bits = 0;
    const int columns_per_pass = rows < kScanThreads ? rows : kScanThreads;
    const int segments = kScanThreads / columns_per_pass;
    const int blocks_per_segment = (num_blocks + segments - 1) / segments;
    for (int column0 = 0; column0 < rows; column0 += columns_per_pass) {
        const int column_local = tid % columns_per_pass;
        const int segment = tid / columns_per_pass;
        const int column = column0 + column_local;
        const bool active = segment < segments && column < rows;
        int32_t* const words = column < experts ? a.histograms + column : reinterpret_cast<int32_t*>(&a.rows->received);
        const int64_t stride = column < experts ? experts : static_cast<int>(sizeof(RowInfo) / sizeof(int32_t));
        const int begin = segment * blocks_per_segment;
        const int end = begin + blocks_per_segment < num_blocks ? begin + blocks_per_segment : num_blocks;
        int sum = 0;
        if (active)
            for (int b = begin; b < end; ++b)
                sum += words[b * stride];
        partial[tid] = active ? sum : 0;
        __syncthreads();
        if (active) {
            int running = 0;
            for (int s = 0; s < segment; ++s)
                running += partial[s * columns_per_pass + column_local];
            for (int b = begin; b < end; ++b) {
                const int count = words[b * stride];
                words[b * stride] = running;
                running += count;
            }
            if (segment == segments - 1)
                column_total[column] = running;
        }
        __syncthreads();
    }

    int bad = 0;
    for (int b = tid; b < num_blocks; b += kScanThreads)
        bad |= a.rows[b].status;
    if (bad)
        atomicOr(&status_bits, bad);

    const int per_thread = (experts + kScanThreads - 1) / kScanThreads;
    const int first = tid * per_thread;
    const int last = first + per_thread < experts ? first + per_thread : experts;
    int64_t padded_sum = 0, count_sum = 0;
    for (int e = first; e < last; ++e) {
        const int64_t count = column_total[e];
        count_sum += count;
        padded_sum += round_up_to(count, a);
    }
    scan[tid] = padded_sum;
    assignments[tid] = count_sum;
    __syncthreads();
    for (int step = 1; step < kScanThreads; step *= 2) {
        const int64_t add_scan = tid >= step ? scan[tid - step] : 0;
        const int64_t add_assign = tid >= step ? assignments[tid - step] : 0;
        __syncthreads();
        scan[tid] += add_scan;
        assignments[tid] += add_assign;
        __syncthreads();
    }
    int64_t running = scan[tid] - padded_sum;
    for (int e = first; e < last; ++e) {
        const int64_t count = column_total[e];
        a.expert_counts[e] = count;
        a.expert_offsets[e] = running;
        running += round_up_to(count, a);
    }
    if (tid == 0) {
        const int64_t received = column_total[experts];
        const int64_t capacity = scan[kScanThreads - 1];
        a.expert_offsets[experts] = capacity;
        a.send_counts[0] = received;
        a.recv_rank_prefix[0] = received;
        a.totals[0] = assignments[kScanThreads - 1];
        publish_counts(a.host_counts, received, capacity, assignments[kScanThreads - 1], status_bits);
    }
}

// Inclusive prefix sum over a wavefront, on the vector unit's own lane shifts (rows of 16, then the
// rows' last lanes): a dozen instructions, against a trip to LDS and back for every step of a shuffle.
template <int kControl, int kRowMask>
__device__ __forceinline__ uint32_t lane_shift(uint32_t value) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(value), kControl, kRowMask, 0xf, false));
}
template <int kControl, int kRowMask>
__device__ __forceinline__ uint64_t lane_shift(uint64_t value) {
    return static_cast<uint64_t>(lane_shift<kControl, kRowMask>(static_cast<uint32_t>(value))) |
           static_cast<uint64_t>(lane_shift<kControl, kRowMask>(static_cast<uint32_t>(value >> 32))) << 32;
}
template <class T>
__device__ __forceinline__ T wave_inclusive_scan(T value) {
    value += lane_shift<0x111, 0xf>(value);  // row_shr:1
    value += lane_shift<0x112, 0xf>(value);
    value += lane_shift<0x114, 0xf>(value);
    value += lane_shift<0x118, 0xf>(value);
    value += lane_shift<0x142, 0xa>(value);  // row_bcast:15 into rows 1 and 3
    value += lane_shift<0x143, 0xc>(value);  // row_bcast:31 into rows 2 and 3
    return value;
}

// One batch of histogram rows of one strip of 64 experts, a wavefront's task: task / strips is the batch,
// task % strips the strip.
struct RowTask {
    uint32_t first_row;
    uint32_t expert;  // this lane's
    uint32_t counts[kSumRows];
};

__device__ __forceinline__ void fetch_rows(const LayoutArgs& a, const PairLane& at, uint32_t task, RowTask& out) {
    const uint32_t batch = fast_divide(task, a.strips_magic, a.strips_shift);
    out.first_row = batch * kSumRows;
    out.expert = (task - batch * a.strips) * kWave + at.lane;
    const uint32_t from = out.expert < a.experts ? out.expert : 0u;
    const int32_t* row = a.histograms + static_cast<uint64_t>(out.first_row) * a.experts;
#pragma unroll
    for (int j = 0; j < kSumRows; ++j) {
        out.counts[j] = static_cast<uint32_t>(row[from]);
        row += a.experts;
    }
}

// (Sums and flags of a wavefront are reduced here before one lane adds them to LDS: an LDS addition of
// different values by all lanes to one word is compiled into a loop over the lanes, a microsecond of it.)
__device__ __forceinline__ uint32_t wave_sum(uint32_t value) { return __builtin_amdgcn_readlane(wave_inclusive_scan(value), kWave - 1); }

// What workgroup 0 of an assignment launch does: it has no tokens; it writes the per-expert outputs and the
// host mailbox (the store to host memory and the wait for it are then on nobody's way to the token writes).
// kDirect: it counts the batch's ids and checks them, with a bit matrix of the whole batch.
template <int kSource>
__device__ __forceinline__ void publish_layout(const LayoutArgs& a, uint32_t* lds) {
    __shared__ uint64_t wave_padded[kLayoutWaves];
    __shared__ RowInfo all;
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const PairLane at = pair_lane(a);
    uint32_t* counts = lds;  // [L]
    uint32_t* bits = lds + (a.experts + 3) / 4 * 4;
    const uint32_t words = kSource == kDirect ? (a.tokens + 31) / 32 : 0u;
    const uint32_t step = a.waves * a.chunk_tokens;
    uint32_t chunk = wave * a.chunk_tokens;
    int64_t id[kChunks];
    if (kSource == kDirect) {
#pragma unroll
        for (int j = 0; j < kChunks; ++j)
            id[j] = fetch_id(a, at, chunk + j * step, a.tokens);
    }
    clear_lds(lds, (a.experts + 3) / 4 * 4 + a.experts * words, a.waves * kWave);
    if (tid == 0)
        all = RowInfo{0, 0, 0, 0};
    __syncthreads();
    uint32_t received = 0, assigned = 0;
    int bad = 0;
    if (kSource == kDirect) {
        while (chunk < a.tokens) {
#pragma unroll
            for (int j = 0; j < kChunks; ++j) {
                const uint32_t chunk_first = chunk + j * step;
                if (chunk_first >= a.tokens)
                    break;
                const bool valid = names_expert(id[j], a);
                const uint64_t valid_mask = __ballot(valid);
                if (valid) {
                    atomicAdd(&counts[static_cast<uint32_t>(id[j])], 1u);
                    if (set_token_bit(bits, words, id[j], chunk_first + at.token))
                        bad |= NANOEP_ROUTING_DUPLICATE;
                }
                bad |= check_id(id[j], a);
                received += count_opening(valid_mask, valid, at);
                assigned += __popcll(valid_mask);
            }
            chunk += kChunks * step;
            if (chunk < a.tokens) {
#pragma unroll
                for (int j = 0; j < kChunks; ++j)
                    id[j] = fetch_id(a, at, chunk + j * step, a.tokens);
            }
        }
    } else {
        for (uint32_t task = wave; task < a.strips * a.row_batches; task += a.waves) {
            RowTask rows;
            fetch_rows(a, at, task, rows);
            uint32_t total = 0;
#pragma unroll
            for (int j = 0; j < kSumRows; ++j)
                total += rows.counts[j];
            if (rows.expert < a.experts)
                atomicAdd(&counts[rows.expert], total);
        }
        for (uint32_t row = tid; row < a.row_count; row += a.waves * kWave) {
            const RowInfo info = a.rows[row];
            received += info.received;
            assigned += info.assigned;
            bad |= info.status;
        }
        received = wave_sum(received);
        assigned = wave_sum(assigned);
    }
    bad = wave_status(bad);
    if (at.lane == 0 && (assigned != 0 || bad != 0)) {
        atomicAdd(&all.received, received);
        atomicAdd(&all.assigned, assigned);
        atomicOr(&all.status, bad);
    }
    __syncthreads();
    const uint32_t first = tid * a.per_thread < a.experts ? tid * a.per_thread : a.experts;
    const uint32_t last = first + a.per_thread < a.experts ? first + a.per_thread : a.experts;
    uint64_t padded_sum = 0, padded_scan = 0;
    if (wave < a.expert_waves) {
        for (uint32_t e = first; e < last; ++e)
            padded_sum += static_cast<uint64_t>(round_up_to(counts[e], a));
        padded_scan = wave_inclusive_scan(padded_sum);
        if (at.lane == kWave - 1)
            wave_padded[wave] = padded_scan;
    }
    __syncthreads();
    if (wave >= a.expert_waves)
        return;
    uint64_t running = padded_scan - padded_sum, capacity = 0;
    for (uint32_t w = 0; w < a.expert_waves; ++w) {
        running += w < wave ? wave_padded[w] : 0u;
        capacity += wave_padded[w];
    }
    if (tid == 0) {
        publish_counts(a.host_counts, all.received, static_cast<int64_t>(capacity), all.assigned, all.status);
        a.expert_offsets[a.experts] = static_cast<int64_t>(capacity);
        a.send_counts[0] = all.received;
        a.recv_rank_prefix[0] = all.received;
        if (a.slot_order != nullptr)
            a.slot_order[a.list_entries] = all.assigned;
    }
    for (uint32_t e = first; e < last; ++e) {
        a.expert_counts[e] = counts[e];
        a.expert_offsets[e] = static_cast<int64_t>(running);
        running += static_cast<uint64_t>(round_up_to(counts[e], a));
    }
}

// Slot assignment.  One workgroup per block of tokens, kOwn chunks of (token, choice) pairs a wavefront, and,
// unless a scan kernel has done that, one more in front of them that publishes (publish_layout).
//
// What a block needs of the others' tokens are sums per expert: the total (for the slots' aligned
// offsets), the part before the block, and the window's part when a window of the slot-order list
// holds several blocks.  kDirect: every workgroup counts the whole batch's ids into LDS by itself, an
// LDS addition a pair, and the layout is one launch.
//
// Nothing here is bound by bytes (the batch's routing is under a megabyte): a launch is 2.2 us, and between
// the first load and the last store lie 2.5 to 3.5 us of round trips and instruction issue: ids and rows
// 0.7 us, counts 0.3, row sums 1.0, expert scan 0.4, slots 0.3, stores 0.7 (4096 x 8, 256 experts).
// Hence a pair a lane instead of a token with all its choices a lane, all loads ahead of the first
// wait, prefix sums by lane shifts in the wavefronts that hold experts only, and 64-token blocks (8
// wavefronts) instead of 256-token ones.  Launch period of the whole layout, before -> after: 16 x 2 5.7 -> 4.8 us,
// 256 x 8 with 64 experts 8.0 -> 5.0, 1537 x 6 with 60 experts 11.0 -> 7.5, 4096 x 8 with 256 experts 12.7 -> 9.0,
// 32768 x 8 with 64 experts 16.1 -> 11.9, with 256 22.5 -> 14.8, 262144 x 4 with 64 experts 91 -> 35; from the call to the
// counts on the host, idle device: 11.5 -> 9.0, 13.0 -> 9.9, 17.0 -> 13.5, 18.1 -> 13.9 us.
//
// The rank of a pair among its block's assignments to the same expert comes from a bit matrix: bit
// (token) of row (expert) is set when the token chose it.  A token's choices are distinct, so the order
// of an expert's assignments is the token order and the rank is the number of bits below the token's.
template <int kSource, bool kWindow, int kOwn>
__global__ void __launch_bounds__(kLayoutThreads) layout_assign_kernel(const LayoutArgs a, const SourceAhead ahead) {
    extern __shared__ __align__(16) uint32_t assign_lds[];
    fetch_layout_arguments(a);
    NANOEP_FETCH_ARGS_2(ahead.x, ahead.work_blocks);
    if (blockIdx.x >= ahead.work_blocks) {
        read_source_ahead(ahead, a.waves);
        return;
    }
    __shared__ uint32_t wave_padded[kLayoutWaves], wave_window[kLayoutWaves];
    __shared__ uint32_t any_bits[kMaxBlockTokens / 32];  // the block's tokens with any valid choice
    __shared__ struct {
        uint32_t received_before;  // tokens with any valid choice before the block
        uint32_t assigned;         // valid choices: all,
        uint32_t assigned_before;  // before the block,
        uint32_t window_start;     // before the window,
        uint32_t own;              // in the block
    } sums;
    if (kSource != kScanned && blockIdx.x == 0) {
        publish_layout<kSource>(a, assign_lds);
        return;
    }
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t block = kSource != kScanned ? blockIdx.x - 1 : blockIdx.x;
    const uint32_t block_first = block * a.block_tokens;
    const uint32_t block_end = block_first + a.block_tokens < a.tokens ? block_first + a.block_tokens : a.tokens;
    const uint32_t window_first = kWindow ? fast_divide(block_first, a.window_magic, a.window_shift) * a.window_tokens : block_first;
    const uint32_t own_row = kSource == kDirect ? 0u : fast_divide(block_first, a.row_magic, a.row_shift);
    const PairLane at = pair_lane(a);
    const uint32_t step = a.waves * a.chunk_tokens;
    // What the workgroup reads leaves before anything waits: the wavefront's own ids, and the first of those it
    // counts: of the whole batch, or what lies between the start of the block's histogram row and the block.
    const uint32_t own_first = block_first + wave * a.chunk_tokens;
    int64_t id[kOwn];
#pragma unroll
    for (int o = 0; o < kOwn; ++o)
        id[o] = fetch_id(a, at, own_first + o * step, block_end);
    const uint32_t count_end = kSource == kDirect ? a.tokens : block_first;
    uint32_t chunk = own_row * a.row_tokens + wave * a.chunk_tokens;
    int64_t batch[kChunks];
#pragma unroll
    for (int j = 0; j < kChunks; ++j)
        batch[j] = fetch_id(a, at, chunk + j * step, count_end);

    const uint32_t tasks = kSource == kSummed ? a.strips * a.row_batches : 0u;
    RowTask rows;
    RowInfo info{0, 0, 0, 0};
    if (kSource == kSummed) {
        fetch_rows(a, at, wave < tasks ? wave : 0u, rows);
        if (tid < a.row_count)
            info = a.rows[tid];
    }

    const uint32_t words = a.block_tokens / 32;
    const uint32_t counter_words = (3 * a.experts + 3) / 4 * 4;
    uint32_t* base = assign_lds;                      // [L] counts before the block -> an expert's first slot in this block
    uint32_t* order_base = base + a.experts;          // [L] the window's counts -> where an expert's run of the list starts
    uint32_t* column_total = order_base + a.experts;  // [L] totals
    uint32_t* bits = assign_lds + counter_words;      // [L][words]
    clear_lds(assign_lds, counter_words + a.experts * words, a.waves * kWave);
    if (tid < kMaxBlockTokens / 32)
        any_bits[tid] = 0;
    if (tid == 0)
        sums = {0, 0, 0, 0, 0};
    __syncthreads();
    uint32_t own = 0;
#pragma unroll
    for (int o = 0; o < kOwn; ++o) {
        const uint32_t own_chunk = own_first + o * step;
        const bool own_valid = names_expert(id[o], a);
        const uint64_t own_mask = __ballot(own_valid);
        const uint32_t local = own_chunk - block_first + at.token;
        if (at.lane < pairs_of_chunk(a, own_chunk, block_end))
            (a.snapshot + static_cast<uint64_t>(own_chunk) * a.topk)[at.lane] = id[o];
        if (own_valid) {
            (void)set_token_bit(bits, words, id[o], local);
            if ((own_mask & at.earlier) == 0)
                atomicOr(&any_bits[local / 32], 1u << (local % 32));
        }
        own += __popcll(own_mask);
    }

    uint32_t received = 0, assigned = 0, before = 0, window_start = 0;
    while (chunk < count_end) {
#pragma unroll
        for (int j = 0; j < kChunks; ++j) {
            const uint32_t chunk_first = chunk + j * step;
            if (chunk_first >= count_end)
                break;  // (the same for the whole wavefront)
            const bool valid = names_expert(batch[j], a);
            const uint64_t valid_mask = __ballot(valid);
            const uint32_t expert = static_cast<uint32_t>(batch[j]);
            const uint32_t token = chunk_first + at.token;
            const bool is_before = kSource != kDirect || token < block_first;
            if (valid) {
                if (kSource == kDirect)
                    atomicAdd(&column_total[expert], is_before ? 0x10001u : 1u);
                else
                    atomicAdd(&base[expert], 1u);
                if (kWindow && (kSource != kDirect || token - window_first < a.window_tokens))
                    atomicAdd(&order_base[expert], kSource != kDirect ? 0x10000u : is_before ? 0x10001u : 1u);
            }
            received += count_opening(valid_mask, valid && is_before, at);
            assigned += __popcll(valid_mask);
            if (kSource == kDirect) {
                before += __popcll(__ballot(valid && is_before));
                if (kWindow)
                    window_start += __popcll(__ballot(valid && token < window_first));
            }
        }
        chunk += kChunks * step;
        if (chunk < count_end) {
#pragma unroll
            for (int j = 0; j < kChunks; ++j)
                batch[j] = fetch_id(a, at, chunk + j * step, count_end);
        }
    }
    if (at.lane == 0) {
        if (own != 0)
            atomicAdd(&sums.own, own);
        if (assigned != 0) {
            atomicAdd(&sums.received_before, received);
            atomicAdd(&sums.assigned_before, kSource == kDirect ? before : assigned);
            if (kSource == kDirect) {
                atomicAdd(&sums.assigned, assigned);
                atomicAdd(&sums.window_start, kWindow ? window_start : before);
            }
        }
    }
    if (kSource == kSummed) {
        const uint32_t window_row = kWindow ? fast_divide(window_first, a.row_magic, a.row_shift) : own_row;
        const uint32_t window_rows = fast_divide(a.window_tokens, a.row_magic, a.row_shift);
        for (uint32_t task = wave; task < tasks; task += a.waves) {
            if (task != wave)
                fetch_rows(a, at, task, rows);
            uint32_t total = 0, earlier = 0, window = 0;
#pragma unroll
            for (int j = 0; j < kSumRows; ++j) {
                const uint32_t row = rows.first_row + j;
                total += rows.counts[j];
                earlier += row < own_row ? rows.counts[j] : 0u;
                if (kWindow)
                    window += row - window_row >= window_rows ? 0u : row < own_row ? rows.counts[j] * 0x10001u : rows.counts[j];
            }
            if (rows.expert < a.experts) {
                atomicAdd(&column_total[rows.expert], total);
                atomicAdd(&base[rows.expert], earlier);
                if (kWindow)
                    atomicAdd(&order_base[rows.expert], window);
            }
        }
        for (uint32_t row = tid; row - at.lane < a.row_count; row += a.waves * kWave) {
            if (row != tid)
                info = row < a.row_count ? a.rows[row] : RowInfo{0, 0, 0, 0};
            const uint32_t all = wave_sum(info.assigned);
            const uint32_t earlier = wave_sum(row < own_row ? info.assigned : 0u);
            const uint32_t earlier_received = wave_sum(row < own_row ? info.received : 0u);
            const uint32_t outside = wave_sum(row < window_row ? info.assigned : 0u);
            if (at.lane == 0) {
                atomicAdd(&sums.assigned, all);
                atomicAdd(&sums.assigned_before, earlier);
                atomicAdd(&sums.received_before, earlier_received);
                atomicAdd(&sums.window_start, outside);
            }
        }
    }
    __syncthreads();
    // Experts: a thread takes a run of them (one each up to the workgroup's threads), the wavefronts
    // without any go on to the last barrier.
    const uint32_t first = tid * a.per_thread < a.experts ? tid * a.per_thread : a.experts;
    const uint32_t last = first + a.per_thread < a.experts ? first + a.per_thread : a.experts;
    // kScanned: exclusive prefixes of the block's row, of the window's first row and of the row behind the
    // window (the totals when there is none)
    const int32_t* prefix_row = a.histograms + static_cast<uint64_t>(own_row) * a.experts;
    const auto padded_of = [&](uint32_t e) -> uint32_t {
        const uint32_t total = kSource == kDirect ? column_total[e] & 0xffffu : column_total[e];
        return kSource == kScanned ? 0u : static_cast<uint32_t>(round_up_to(total, a));
    };
    const auto before_of = [&](uint32_t e) -> uint32_t {
        return kSource == kDirect ? column_total[e] >> 16 : kSource == kSummed ? base[e] : base[e] + static_cast<uint32_t>(prefix_row[e]);
    };
    // the window's assignments to the expert, and those of them in the blocks before this one << 16
    const auto window_of = [&](uint32_t e) -> uint32_t {
        if (!kWindow) {
            uint32_t count = 0;
            for (uint32_t w = 0; w < words; ++w)
                count += __popc(bits[e * words + w]);
            return count;
        }
        if (kSource != kScanned)
            return order_base[e];
        const uint32_t first_row = fast_divide(window_first, a.row_magic, a.row_shift);
        const uint32_t end_row = first_row + fast_divide(a.window_tokens, a.row_magic, a.row_shift);
        const uint32_t at_first = static_cast<uint32_t>(a.histograms[static_cast<uint64_t>(first_row) * a.experts + e]);
        const uint32_t at_end = end_row < a.row_count ? static_cast<uint32_t>(a.histograms[static_cast<uint64_t>(end_row) * a.experts + e])
                                                      : static_cast<uint32_t>(a.expert_counts[e]);
        return order_base[e] + (at_end - at_first) + ((static_cast<uint32_t>(prefix_row[e]) - at_first) << 16);
    };
    uint32_t padded_sum = 0, padded_scan = 0, window_sum = 0, window_scan = 0;
    if (wave < a.expert_waves) {
        uint32_t before_sum = 0, window_before_sum = 0;
        for (uint32_t e = first; e < last; ++e) {
            const uint32_t window = window_of(e);
            padded_sum += padded_of(e);
            window_sum += window & 0xffffu;
            if (kSource == kScanned) {
                before_sum += before_of(e);
                window_before_sum += window >> 16;
            }
        }
        padded_scan = wave_inclusive_scan(padded_sum);
        window_scan = wave_inclusive_scan(window_sum);
        if (at.lane == kWave - 1) {
            wave_padded[wave] = padded_scan;
            wave_window[wave] = window_scan;
        }
        if (kSource == kScanned) {
            // (the rows' sums: the partial row's are in already)
            before_sum = wave_inclusive_scan(before_sum);
            window_before_sum = wave_inclusive_scan(window_before_sum);
            if (at.lane == kWave - 1) {
                atomicAdd(&sums.assigned, before_sum);
                atomicAdd(&sums.window_start, before_sum - window_before_sum);
            }
        }
    }
    if (a.expert_waves > 1)
        __syncthreads();
    else
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the sums stay within the one wavefront
    if (wave < a.expert_waves) {
        uint32_t running = padded_scan - padded_sum;
        uint32_t running_window = window_scan - window_sum + sums.window_start;  // the list is dense
        for (uint32_t w = 0; w < wave; ++w) {
            running += wave_padded[w];
            running_window += wave_window[w];
        }
        for (uint32_t e = first; e < last; ++e) {
            const uint32_t window = window_of(e), padded = padded_of(e);
            base[e] = (kSource == kScanned ? static_cast<uint32_t>(a.expert_offsets[e]) : running) + before_of(e);
            order_base[e] = running_window + (window >> 16);  // behind the expert's entries of the window's earlier blocks
            running += padded;
            running_window += window & 0xffffu;
        }
    }
    __syncthreads();
    if (kSource == kScanned && tid == 0) {
        sums.assigned_before = sums.assigned;
        sums.assigned = static_cast<uint32_t>(a.totals[0]);
        sums.received_before += a.rows[own_row].received;
    }
    if (kSource == kScanned)
        __syncthreads();

#pragma unroll
    for (int o = 0; o < kOwn; ++o) {
        const uint32_t own_chunk = own_first + o * step;
        if (at.lane >= pairs_of_chunk(a, own_chunk, block_end))
            continue;
        const uint32_t local = own_chunk - block_first + at.token;
        const uint32_t token = own_chunk + at.token;
        const uint32_t word = local / 32, below = (1u << (local % 32)) - 1u;
        int32_t value = -1;
        if (names_expert(id[o], a)) {
            const uint32_t expert = static_cast<uint32_t>(id[o]);
            uint32_t rank = 0;
            for (uint32_t w = 0; w < words; ++w) {
                const uint32_t row = bits[expert * words + w];
                rank += __popc(w < word ? row : w == word ? row & below : 0u);
            }
            value = a.expand ? static_cast<int32_t>(base[expert] + rank) : static_cast<int32_t>(expert);
            if (a.slot_order != nullptr)
                a.slot_order[order_base[expert] + rank] =
                    static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint32_t>(value)) << 32 | (own_chunk * a.topk + at.lane));
        }
        if (a.token_slots != nullptr)
            (a.token_slots + static_cast<uint64_t>(own_chunk) * a.topk)[at.lane] = value;
        const bool is_received = (any_bits[word] >> (local % 32)) & 1u;
        uint32_t row = sums.received_before;
        for (uint32_t w = 0; w < words; ++w)
            row += __popc(w < word ? any_bits[w] : w == word ? any_bits[w] & below : 0u);
        if (at.k == 0)
            a.dst_slots[token] = is_received ? static_cast<int64_t>(row) : -1;
        if (is_received) {
            // the receive row [0, token, K values]
            int32_t* out = a.recv_metadata + static_cast<uint64_t>(row) * (a.topk + 2);
            out[2 + at.k] = value;
            if (at.k == 0) {
                out[0] = 0;
                out[1] = static_cast<int32_t>(token);
            }
        }
    }
    if (a.slot_order != nullptr) {
        // every block clears as many entries of the list's unused tail as it has masked choices; the last one
        // also what lies behind the batch's own entries, so that everything from entry A to the count word reads -1
        const uint64_t entries_before = static_cast<uint64_t>(block_first) * a.topk;
        int64_t* tail = a.slot_order + sums.assigned + (entries_before - sums.assigned_before);
        const uint32_t holes = (block_end - block_first) * a.topk - sums.own;
        for (uint32_t i = tid; i < holes; i += a.waves * kWave)
            tail[i] = -1;
        if (block == a.blocks - 1)
            for (uint64_t i = static_cast<uint64_t>(a.tokens) * a.topk + tid; i < a.list_entries; i += a.waves * kWave)
                a.slot_order[i] = -1;
        if (kSource == kScanned && block == 0 && tid == 0)
            a.slot_order[a.list_entries] = sums.assigned;
    }
}

// Argument checks shared by the two layout entry points (everything but the workspace).
int check_layout_arguments(const int64_t* topk_idx, int64_t num_tokens, int num_topk, int64_t num_local_experts, int64_t alignment,
                           int expand, int hidden, const int32_t* recv_metadata, const int64_t* expert_counts,
                           const int64_t* expert_offsets, const int64_t* dst_slots, const int64_t* send_counts,
                           const int64_t* topk_snapshot, const int64_t* recv_rank_prefix, const int64_t* slot_order,
                           const int64_t* host_counts) {
    if (num_tokens < 0 || num_tokens > INT32_MAX || num_topk <= 0 || num_topk > kMaxTopk || num_local_experts <= 0 ||
        !layout_supports(num_local_experts) || alignment <= 0 || alignment > (int64_t{1} << 31) || hidden < 0)
        return NANOEP_ERR_INVALID_ARGUMENT;
    if (expert_counts == nullptr || expert_offsets == nullptr || send_counts == nullptr || recv_rank_prefix == nullptr ||
        host_counts == nullptr)
        return NANOEP_ERR_INVALID_ARGUMENT;
    if (num_tokens > 0 && (topk_idx == nullptr || recv_metadata == nullptr || dst_slots == nullptr || topk_snapshot == nullptr))
        return NANOEP_ERR_INVALID_ARGUMENT;
    // the slot-order list packs token * K + k into 32 bits and only exists for the expanded layout
    if (slot_order != nullptr && (!expand || num_tokens * num_topk >= (int64_t{1} << 31)))
        return NANOEP_ERR_INVALID_ARGUMENT;
    return NANOEP_OK;
}

// The launches of one layout, from the batch's geometry.
struct LayoutPlan {
    int window;
    int block_tokens;
    int64_t blocks;
    int histogram_tokens;
    int64_t histogram_rows;
    int source;
    int chunk_tokens;
    int own;            // chunks of its block an assignment wavefront takes
    int waves;          // of an assignment workgroup
    int row_waves;      // of a histogram workgroup
    size_t assign_lds;
    // workgroups of the two launches, without those that read ahead
    uint32_t row_blocks;
    uint32_t assign_blocks;
    // ... and those that do where the rows are known
    AheadPlan beside_rows;
    AheadPlan beside_assignment;
};

LayoutPlan plan_layout(int64_t num_tokens, int num_topk, int64_t num_local_experts, int hidden, const Knobs& knobs) {
    LayoutPlan plan{};
    plan.window = layout_window_tokens(num_tokens, hidden, knobs);
    plan.block_tokens = layout_block_tokens_of(num_tokens, plan.window, num_topk, num_local_experts);
    plan.blocks = (num_tokens + plan.block_tokens - 1) / plan.block_tokens;
    plan.histogram_tokens = layout_histogram_tokens(num_tokens, plan.window, plan.block_tokens, num_topk, num_local_experts);
    plan.histogram_rows = (num_tokens + plan.histogram_tokens - 1) / plan.histogram_tokens;

    const int64_t pairs = num_tokens * num_topk;
    const int64_t batch_words = (num_tokens + 31) / 32;
    const int64_t block_words = plan.block_tokens / 32;
    const size_t direct_lds = layout_lds(num_local_experts, batch_words > block_words ? batch_words : block_words);
    const bool direct_fits = pairs < 65536 && direct_lds <= kLayoutLdsBudget;
    plan.source = direct_fits && pairs <= kDirectPairs ? kDirect : plan.histogram_rows <= kSummedHistograms ? kSummed : kScanned;
    if (knobs.layout_launches == 1 && direct_fits)
        plan.source = kDirect;
    else if (knobs.layout_launches == 2 && num_tokens > 0)
        plan.source = kSummed;
    else if (knobs.layout_launches == 3)
        plan.source = kScanned;
    plan.assign_lds = plan.source == kDirect ? direct_lds : layout_lds(num_local_experts, block_words);
    // one or more chunks of the block a wavefront; in the direct plan enough wavefronts for the counting as well
    plan.chunk_tokens = kWave / num_topk;
    int waves = (plan.block_tokens + plan.chunk_tokens - 1) / plan.chunk_tokens;
    if (plan.source == kDirect) {
        const int64_t counting = (pairs / kChunks + kWave - 1) / kWave;
        if (num_tokens < plan.block_tokens)
            waves = static_cast<int>((num_tokens + plan.chunk_tokens - 1) / plan.chunk_tokens);
        if (waves < counting)
            waves = counting < kLayoutWaves ? static_cast<int>(counting) : kLayoutWaves;
    }
    plan.own = plan.source == kScanned ? kScannedChunks : plan.source == kSummed && plan.blocks * waves > kOneChunkWaves ? kSummedChunks : 1;
    waves = (waves + plan.own - 1) / plan.own;
    if (plan.source == kSummed) {
        const int64_t tasks = (num_local_experts + kWave - 1) / kWave * (padded_rows(plan.histogram_rows) / kSumRows);
        if (waves < tasks)
            waves = tasks < 8 ? static_cast<int>(tasks) : waves < 8 ? 8 : waves;
    }
    plan.waves = waves < 2 ? 2 : waves;
    const int row_waves = (plan.histogram_tokens + plan.chunk_tokens - 1) / plan.chunk_tokens;
    plan.row_waves = row_waves < 2 ? 2 : row_waves > kLayoutWaves ? kLayoutWaves : row_waves;
    plan.row_blocks = static_cast<uint32_t>(padded_rows(plan.histogram_rows));
    plan.assign_blocks = static_cast<uint32_t>(plan.blocks + (plan.source == kScanned ? 0 : 1));

    const int64_t row_vectors = hidden / 8, xcds = make_xcd_map(knobs.xcds).count;
    if (plan.source != kDirect && pairs >= kHistogramAheadPairs)
        plan.beside_rows = plan_ahead(num_tokens, row_vectors, plan.window, xcds, plan.row_waves, kHistogramAheadBytes);
    else
        plan.beside_assignment = plan_ahead(num_tokens, row_vectors, plan.window, xcds, plan.waves, kAssignAheadBytes);
    const auto launched = [&] { return static_cast<int64_t>(plan.assign_blocks) + plan.beside_assignment.blocks; };
    if (launched() * 4 > knobs.cus * int64_t{3})
        plan.beside_assignment = plan_ahead(num_tokens, row_vectors, plan.window, xcds, plan.waves, kAssignAheadBytes / 2);
    if (launched() > knobs.cus)
        plan.beside_assignment = {0, 0, 0};
    return plan;
}

// Enqueues the layout launches over a carved workspace; the arguments have been checked.  x: the rows that will be
// dispatched right behind the layout, or null.
int enqueue_layout(const int64_t* topk_idx, int64_t num_tokens, int num_topk, int64_t num_local_experts, int64_t alignment,
                   int expand, int hidden, int32_t* recv_metadata, int64_t* expert_counts, int64_t* expert_offsets,
                   int64_t* dst_slots, int64_t* send_counts, int64_t* topk_snapshot, int64_t* recv_rank_prefix,
                   int32_t* token_slots, int64_t* slot_order, const LayoutWorkspace& ws, int64_t* host_counts,
                   const void* x, void* stream_handle, const Knobs& knobs) {
    const LayoutPlan plan = plan_layout(num_tokens, num_topk, num_local_experts, hidden, knobs);
    int check_tokens = plan.histogram_tokens;
    while (check_tokens > plan.block_tokens && layout_lds(num_local_experts, check_tokens / 32) > kLayoutLdsBudget)
        check_tokens = plan.block_tokens;
    auto stream = static_cast<hipStream_t>(stream_handle);
    const int threads = plan.waves * kWave;

    const FastDivisor alignment_divisor = make_fast_divisor(static_cast<uint32_t>(alignment));
    const FastDivisor row_divisor = make_fast_divisor(static_cast<uint32_t>(plan.histogram_tokens));
    const FastDivisor window_divisor = make_fast_divisor(static_cast<uint32_t>(plan.window));
    LayoutArgs a{};
    a.topk_idx = topk_idx;
    a.histograms = ws.histograms;
    a.rows = ws.rows;
    a.tokens = static_cast<uint32_t>(num_tokens);
    a.topk = static_cast<uint32_t>(num_topk);
    a.experts = static_cast<uint32_t>(num_local_experts);
    a.chunk_tokens = static_cast<uint32_t>(plan.chunk_tokens);
    a.chunk_pairs = a.chunk_tokens * a.topk;
    a.topk_magic = (65536u + a.topk - 1) / a.topk;
    a.waves = static_cast<uint32_t>(plan.waves);
    a.block_tokens = static_cast<uint32_t>(plan.block_tokens);
    a.row_tokens = static_cast<uint32_t>(plan.histogram_tokens);
    a.row_magic = row_divisor.magic;
    a.row_shift = row_divisor.shift;
    a.window_tokens = static_cast<uint32_t>(plan.window);
    a.window_magic = window_divisor.magic;
    a.window_shift = window_divisor.shift;
    a.row_count = static_cast<uint32_t>(plan.histogram_rows);
    a.row_batches = plan.row_blocks / kSumRows;
    a.strips = (a.experts + kWave - 1) / kWave;
    const FastDivisor strips_divisor = make_fast_divisor(a.strips);
    a.strips_magic = strips_divisor.magic;
    a.strips_shift = strips_divisor.shift;
    a.per_thread = (a.experts + threads - 1) / threads;
    a.expert_waves = ((a.experts + a.per_thread - 1) / a.per_thread + kWave - 1) / kWave;
    a.check_tokens = static_cast<uint32_t>(check_tokens);
    a.expand = expand ? 1u : 0u;
    a.alignment = alignment;
    a.alignment_magic = alignment_divisor.magic;
    a.alignment_shift = alignment_divisor.shift;
    a.totals = ws.totals;
    a.expert_counts = expert_counts;
    a.expert_offsets = expert_offsets;
    a.send_counts = send_counts;
    a.recv_rank_prefix = recv_rank_prefix;
    a.host_counts = host_counts;
    a.snapshot = topk_snapshot;
    a.recv_metadata = recv_metadata;
    a.dst_slots = dst_slots;
    a.token_slots = token_slots;
    a.slot_order = num_tokens > 0 ? slot_order : nullptr;
    a.list_entries = static_cast<uint64_t>((num_tokens + kOrderTokens - 1) / kOrderTokens * kOrderTokens) * num_topk;
    a.blocks = static_cast<uint32_t>(plan.blocks);

    SourceAhead ahead{};
    ahead.x = static_cast<const u32x4*>(x);
    ahead.xcds = make_xcd_map(knobs.xcds);
    // Workgroups of a launch with those that read ahead.
    const auto with_ahead = [&](uint32_t work_blocks, const AheadPlan& beside) {
        ahead.work_blocks = work_blocks;
        ahead.vectors = beside.vectors;
        ahead.share = beside.share;
        return work_blocks + (x == nullptr ? 0u : beside.blocks);
    };

    __atomic_store_n(&host_counts[0], int64_t{-1}, __ATOMIC_RELEASE);
    if (plan.source != kDirect && plan.histogram_rows > 0) {
        const uint32_t grid = with_ahead(plan.row_blocks, plan.beside_rows);
        layout_histogram_kernel<<<grid, plan.row_waves * kWave, layout_lds(num_local_experts, check_tokens / 32), stream>>>(
            a, static_cast<uint32_t>(plan.row_waves), ahead);
        NANOEP_HIP_TRY(hipGetLastError());
    }
    if (plan.source == kScanned) {
        layout_scan_kernel<<<1, kScanThreads, static_cast<size_t>(num_local_experts + 1) * 4, stream>>>(a);
        NANOEP_HIP_TRY(hipGetLastError());
        if (plan.blocks == 0)
            return NANOEP_OK;
    }
    const dim3 grid(with_ahead(plan.assign_blocks, plan.beside_assignment));
    const bool several = plan.window > plan.block_tokens;
#define NANOEP_LAUNCH_ASSIGN(SOURCE, OWN)                                                       \
    do {                                                                                        \
        if (several)                                                                            \
            layout_assign_kernel<SOURCE, true, OWN><<<grid, threads, plan.assign_lds, stream>>>(a, ahead);  \
        else                                                                                    \
            layout_assign_kernel<SOURCE, false, OWN><<<grid, threads, plan.assign_lds, stream>>>(a, ahead); \
    } while (0)
    if (plan.source == kDirect)
        NANOEP_LAUNCH_ASSIGN(kDirect, 1);
    else if (plan.source == kSummed && plan.own == 1)
        NANOEP_LAUNCH_ASSIGN(kSummed, 1);
    else if (plan.source == kSummed)
        NANOEP_LAUNCH_ASSIGN(kSummed, kSummedChunks);
    else
        NANOEP_LAUNCH_ASSIGN(kScanned, kScannedChunks);
#undef NANOEP_LAUNCH_ASSIGN
    NANOEP_HIP_TRY(hipGetLastError());
    return NANOEP_OK;
}

// ---- The private handle tensors rebuilt from a handle's own public ones -------------------------
//
// A handle that went through a caller keeping only the reference's seven tensors has lost the slot
// table and the slot-order list.  Both are functions of dst_slots and recv_metadata alone:
// token_slots[t][k] = recv_metadata[dst_slots[t]][2 + k] (-1 when the token was not sent or the slot
// lies outside [0, C)), and the list is, window of consecutive tokens by window, the valid (slot,
// t * K + k) pairs in ascending slot order.  Nothing here looks at the routing ids or assumes the
// slots were made by this library: the handle is followed as it is written.

// Largest number of list entries one window may hold here: the sort runs in LDS, 8 bytes an entry.
constexpr int kRebuildMaxWindowEntries = 4096;
constexpr int kRebuildThreads = 1024;

// Tokens of one window of a rebuilt list: the layout's own choice for this batch, halved until a
// window's T * K entries fit the sort.
int rebuild_window_tokens(int64_t tokens_total, int num_topk, int hidden, const Knobs& knobs) {
    int window = layout_window_tokens(tokens_total, hidden, knobs);
    if (window > kMaxWindowTokens)
        window = kMaxWindowTokens;
    while (window > 32 && static_cast<int64_t>(window) * num_topk > kRebuildMaxWindowEntries)
        window /= 2;
    return window;
}

// One workgroup per window: the slot table of the window's tokens and the number of valid entries.
__global__ void __launch_bounds__(kRebuildThreads) rebuild_table_kernel(const int32_t* __restrict__ recv_metadata,  // [N][K+2]
                                                                       const int64_t* __restrict__ dst_slots,     // [T]
                                                                       int64_t recv_count,
                                                                       int64_t out_rows,
                                                                       int64_t num_tokens,
                                                                       int num_topk,
                                                                       int window_tokens,
                                                                       int32_t* __restrict__ token_slots,  // [T][K]
                                                                       int32_t* __restrict__ window_counts) {
    __shared__ int valid_entries;
    if (threadIdx.x == 0)
        valid_entries = 0;
    __syncthreads();
    const int64_t first = static_cast<int64_t>(blockIdx.x) * window_tokens * num_topk;
    const int64_t batch_end = num_tokens * num_topk;
    const int64_t window_end = first + static_cast<int64_t>(window_tokens) * num_topk;
    const int64_t end = window_end < batch_end ? window_end : batch_end;
    int mine = 0;
    for (int64_t flat = first + threadIdx.x; flat < end; flat += kRebuildThreads) {
        const int64_t token = flat / num_topk;
        const int k = static_cast<int>(flat - token * num_topk);
        const int64_t row = dst_slots[token];
        int32_t slot = -1;
        if (row >= 0 && row < recv_count)
            slot = recv_metadata[row * (num_topk + 2) + 2 + k];
        if (slot < 0 || slot >= out_rows)
            slot = -1;
        token_slots[flat] = slot;
        mine += slot >= 0;
    }
#pragma unroll
    for (int distance = kWave / 2; distance > 0; distance /= 2)
        mine += __shfl_xor(mine, distance, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0 && mine != 0)
        atomicAdd(&valid_entries, mine);
    __syncthreads();
    if (threadIdx.x == 0)
        window_counts[blockIdx.x] = valid_entries;
}

// One workgroup per window: sorts the window's (slot, source) pairs in LDS (bitonic network over
// `sort_size` keys, a power of two; masked choices sort behind everything as the largest key) and
// writes the valid ones where the list has room for them: behind the entries of all earlier
// windows.  The rest of the buffer reads -1 up to the count word, as the layout leaves it.
__global__ void __launch_bounds__(kRebuildThreads) rebuild_order_kernel(const int32_t* __restrict__ token_slots,    // [T][K]
                                                                       const int32_t* __restrict__ window_counts,  // [windows]
                                                                       int64_t num_tokens,
                                                                       int num_topk,
                                                                       int window_tokens,
                                                                       int num_windows,
                                                                       int sort_size,
                                                                       int64_t* __restrict__ slot_order,
                                                                       int64_t capacity_entries,
                                                                       int64_t* host_count,  // pinned, or null
                                                                       int64_t host_tag) {
    extern __shared__ int64_t sort_keys[];
    __shared__ int64_t before_sum;
    __shared__ int64_t total_sum;
    const int window = blockIdx.x;
    const int tid = threadIdx.x;
    if (tid == 0) {
        before_sum = 0;
        total_sum = 0;
    }
    const int64_t first = static_cast<int64_t>(window) * window_tokens * num_topk;
    const int64_t batch_end = num_tokens * num_topk;
    const int64_t window_end = first + static_cast<int64_t>(window_tokens) * num_topk;
    const int64_t end = window_end < batch_end ? window_end : batch_end;
    for (int i = tid; i < sort_size; i += kRebuildThreads) {
        const int64_t flat = first + i;
        int64_t key = INT64_MAX;
        if (flat < end) {
            const int32_t slot = token_slots[flat];
            if (slot >= 0)
                key = (static_cast<int64_t>(slot) << 32) | static_cast<int64_t>(static_cast<uint32_t>(flat));
        }
        sort_keys[i] = key;
    }
    __syncthreads();
    // valid entries of the windows before this one, and of all windows
    int64_t before = 0, total = 0;
    for (int w = tid; w < num_windows; w += kRebuildThreads) {
        const int count = window_counts[w];
        total += count;
        before += w < window ? count : 0;
    }
#pragma unroll
    for (int distance = kWave / 2; distance > 0; distance /= 2) {
        before += __shfl_xor(before, distance, kWave);
        total += __shfl_xor(total, distance, kWave);
    }
    if ((tid & (kWave - 1)) == 0 && total != 0) {
        atomicAdd(reinterpret_cast<unsigned long long*>(&before_sum), static_cast<unsigned long long>(before));
        atomicAdd(reinterpret_cast<unsigned long long*>(&total_sum), static_cast<unsigned long long>(total));
    }
    for (int size = 2; size <= sort_size; size *= 2) {
        for (int stride = size / 2; stride > 0; stride /= 2) {
            for (int i = tid; i < sort_size; i += kRebuildThreads) {
                const int partner = i ^ stride;
                if (partner > i) {
                    const bool ascending = (i & size) == 0;
                    const int64_t a = sort_keys[i], b = sort_keys[partner];
                    if ((a > b) == ascending) {
                        sort_keys[i] = b;
                        sort_keys[partner] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
    __syncthreads();
    const int64_t assigned_before = before_sum;
    const int64_t assigned = total_sum;
    const int own = window_counts[window];
    for (int i = tid; i < own; i += kRebuildThreads)
        slot_order[assigned_before + i] = sort_keys[i];
    // the unused tail: every window clears as many entries as it has masked choices, the last one also
    // what lies between the batch's last choice and the count word
    const int64_t own_entries = end - first;
    int64_t* tail = slot_order + assigned + (first - assigned_before);
    for (int64_t i = tid; i < own_entries - own; i += kRebuildThreads)
        tail[i] = -1;
    if (window == num_windows - 1) {
        for (int64_t i = batch_end + tid; i < capacity_entries; i += kRebuildThreads)
            slot_order[i] = -1;
        if (tid == 0) {
            slot_order[capacity_entries] = assigned;
            if (host_count != nullptr) {
                __threadfence_system();
                __hip_atomic_store(host_count, host_tag | assigned, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    }
}

// Address of this file's `scratch` array on the current device, resolved once per device (each GPU
// holds its own copy at its own address).
constexpr int kMaxDevices = 64;
std::mutex g_static_scratch_mutex;
void* g_static_scratch[kMaxDevices] = {};

int static_scratch_of_current_device(void** out) {
    int device = -1;
    NANOEP_HIP_TRY(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices)
        return NANOEP_ERR_INVALID_ARGUMENT;
    std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
    if (g_static_scratch[device] == nullptr) {
        void* address = nullptr;
        NANOEP_HIP_TRY(hipGetSymbolAddress(&address, HIP_SYMBOL(scratch)));
        if (address == nullptr)
            return NANOEP_ERR_HIP;
        g_static_scratch[device] = address;
    }
    *out = g_static_scratch[device];
    return NANOEP_OK;
}

// Whether nanoep_dispatch walks the slot-order list of such a batch, and sources are read ahead of their copies at all.
bool list_walk_follows(int64_t num_tokens, int num_topk, int64_t num_local_experts, int hidden) {
    const Tuning tuning = current_tuning();
    return num_tokens * num_topk < (int64_t{1} << 31) && tuning.dispatch_prefetch != 0 &&
           plan_list_walk(num_tokens, nanoep_slot_order_entries(num_tokens, num_topk, num_local_experts) - 1, hidden, tuning).taken;
}

}  // namespace
}  // namespace nanoep

using namespace nanoep;

extern "C" {

size_t nanoep_layout_workspace_bytes(int64_t num_tokens, int num_topk, int64_t num_local_experts) {
    if (num_tokens < 0 || num_topk <= 0 || num_local_experts <= 0)
        return 0;
    return carve_layout_workspace(nullptr, num_tokens, num_topk, num_local_experts, current_knobs()).bytes;
}

int nanoep_layout_block_tokens(int64_t num_tokens, int64_t num_local_experts, int hidden) {
    if (num_local_experts <= 0 || num_tokens < 0 || hidden < 0)
        return 0;
    return layout_supports(num_local_experts) ? layout_window_tokens(num_tokens, hidden, current_knobs()) : 0;
}

int64_t nanoep_layout_ahead_bytes(int64_t num_tokens, int num_topk, int64_t num_local_experts, int hidden) {
    if (num_tokens <= 0 || num_tokens > INT32_MAX || num_topk <= 0 || num_topk > kMaxTopk || !layout_supports(num_local_experts) || hidden <= 0 ||
        hidden % 8 != 0)
        return 0;
    const Knobs knobs = current_knobs();
    if (!list_walk_follows(num_tokens, num_topk, num_local_experts, hidden))
        return 0;
    const LayoutPlan plan = plan_layout(num_tokens, num_topk, num_local_experts, hidden, knobs);
    const uint32_t xcds = make_xcd_map(knobs.xcds).count;
    return ahead_bytes(plan.beside_rows, plan.row_blocks, xcds, plan.row_waves) +
           ahead_bytes(plan.beside_assignment, plan.assign_blocks, xcds, plan.waves);
}

int64_t nanoep_slot_order_entries(int64_t num_tokens, int num_topk, int64_t num_local_experts) {
    if (num_tokens < 0 || num_topk <= 0 || num_local_experts <= 0)
        return 0;
    if (!layout_supports(num_local_experts) || num_tokens == 0)
        return 0;
    return (num_tokens + kOrderTokens - 1) / kOrderTokens * kOrderTokens * num_topk + 1;  // the count word last
}

int nanoep_layout(const int64_t* topk_idx, int64_t num_tokens, int num_topk, int64_t num_local_experts,
                  int64_t alignment, int expand, int hidden, int32_t* recv_metadata, int64_t* expert_counts,
                  int64_t* expert_offsets, int64_t* dst_slots, int64_t* send_counts, int64_t* topk_snapshot,
                  int64_t* recv_rank_prefix, int32_t* token_slots, int64_t* slot_order, void* workspace,
                  size_t workspace_bytes, int64_t* host_counts, void* stream_handle) {
    return nanoep_layout_ahead(topk_idx, num_tokens, num_topk, num_local_experts, alignment, expand, hidden, recv_metadata,
                               expert_counts, expert_offsets, dst_slots, send_counts, topk_snapshot, recv_rank_prefix, token_slots,
                               slot_order, workspace, workspace_bytes, host_counts, nullptr, stream_handle);
}

int nanoep_layout_ahead(const int64_t* topk_idx, int64_t num_tokens, int num_topk, int64_t num_local_experts,
                        int64_t alignment, int expand, int hidden, int32_t* recv_metadata, int64_t* expert_counts,
                        int64_t* expert_offsets, int64_t* dst_slots, int64_t* send_counts, int64_t* topk_snapshot,
                        int64_t* recv_rank_prefix, int32_t* token_slots, int64_t* slot_order, void* workspace,
                        size_t workspace_bytes, int64_t* host_counts, const void* x, void* stream_handle) {
    const Knobs knobs = current_knobs();
    const int status = check_layout_arguments(topk_idx, num_tokens, num_topk, num_local_experts, alignment, expand, hidden,
                                              recv_metadata, expert_counts, expert_offsets, dst_slots, send_counts, topk_snapshot,
                                              recv_rank_prefix, slot_order, host_counts);
    if (status != NANOEP_OK)
        return status;
    if (workspace == nullptr || (x != nullptr && (hidden % 8 != 0 || !aligned16(x))))
        return NANOEP_ERR_INVALID_ARGUMENT;
    const LayoutWorkspace ws = carve_layout_workspace(workspace, num_tokens, num_topk, num_local_experts, knobs);
    if (ws.bytes > workspace_bytes)
        return NANOEP_ERR_WORKSPACE;
    const bool ahead = x != nullptr && slot_order != nullptr && list_walk_follows(num_tokens, num_topk, num_local_experts, hidden);
    return enqueue_layout(topk_idx, num_tokens, num_topk, num_local_experts, alignment, expand, hidden, recv_metadata, expert_counts,
                          expert_offsets, dst_slots, send_counts, topk_snapshot, recv_rank_prefix, token_slots, slot_order, ws,
                          host_counts, ahead ? x : nullptr, stream_handle, knobs);
}

int nanoep_layout_static(const int64_t* topk_idx, int64_t num_tokens, int num_topk, int64_t num_local_experts,
                         int64_t alignment, int expand, int hidden, int32_t* recv_metadata, int64_t* expert_counts,
                         int64_t* expert_offsets, int64_t* dst_slots, int64_t* send_counts, int64_t* topk_snapshot,
                         int64_t* recv_rank_prefix, int32_t* token_slots, int64_t* slot_order, int64_t* host_counts,
                         void* stream_handle) {
    const Knobs knobs = current_knobs();
    const int status = check_layout_arguments(topk_idx, num_tokens, num_topk, num_local_experts, alignment, expand, hidden,
                                              recv_metadata, expert_counts, expert_offsets, dst_slots, send_counts, topk_snapshot,
                                              recv_rank_prefix, slot_order, host_counts);
    if (status != NANOEP_OK)
        return status;
    // the size is checked before any device is touched
    if (carve_layout_workspace(nullptr, num_tokens, num_topk, num_local_experts, knobs).bytes > NANOEP_STATIC_SCRATCH_BYTES)
        return NANOEP_ERR_SCRATCH_LIMIT;
    void* base = nullptr;
    const int scratch_status = static_scratch_of_current_device(&base);
    if (scratch_status != NANOEP_OK)
        return scratch_status;
    // Nothing in the workspace has to start at zero: the histogram kernel writes every row (counts
    // and status) that the later kernels of the same call read.
    const LayoutWorkspace ws = carve_layout_workspace(base, num_tokens, num_topk, num_local_experts, knobs);
    return enqueue_layout(topk_idx, num_tokens, num_topk, num_local_experts, alignment, expand, hidden, recv_metadata, expert_counts,
                          expert_offsets, dst_slots, send_counts, topk_snapshot, recv_rank_prefix, token_slots, slot_order, ws,
                          host_counts, nullptr, stream_handle, knobs);
}

size_t nanoep_rebuild_workspace_bytes(int64_t num_tokens, int num_topk) {
    if (num_tokens < 0 || num_topk <= 0 || num_topk > kMaxTopk)
        return 0;
    // one int32 per window of the smallest size a rebuilt list takes
    return align_up(static_cast<size_t>((num_tokens + 31) / 32) * 4, 256) + 256;
}

int nanoep_rebuild_window_tokens(int64_t num_tokens, int num_topk, int hidden) {
    if (num_tokens < 0 || num_topk <= 0 || num_topk > kMaxTopk || hidden < 0)
        return 0;
    return rebuild_window_tokens(num_tokens, num_topk, hidden, current_knobs());
}

int nanoep_rebuild_order(const int32_t* recv_metadata, const int64_t* dst_slots, int64_t recv_count, int64_t expanded_capacity,
                         int64_t num_tokens, int num_topk, int64_t num_local_experts, int hidden, int32_t* token_slots,
                         int64_t* slot_order, void* workspace, size_t workspace_bytes, int64_t* host_count, int64_t host_tag,
                         void* stream_handle) {
    if (num_tokens <= 0 || num_tokens > INT32_MAX || num_topk <= 0 || num_topk > kMaxTopk || num_local_experts <= 0 || hidden < 0 ||
        recv_count < 0 || recv_count > num_tokens || expanded_capacity < 0 || expanded_capacity > INT32_MAX ||
        num_tokens * num_topk >= (int64_t{1} << 31))
        return NANOEP_ERR_INVALID_ARGUMENT;
    if (dst_slots == nullptr || token_slots == nullptr || slot_order == nullptr || workspace == nullptr ||
        (recv_count > 0 && recv_metadata == nullptr) || host_tag < 0 || (host_tag & 0xffffffffll) != 0)
        return NANOEP_ERR_INVALID_ARGUMENT;
    const Knobs knobs = current_knobs();
    if (!layout_supports(num_local_experts))
        return NANOEP_ERR_INVALID_ARGUMENT;  // no slot-order buffer exists for this geometry
    if (nanoep_rebuild_workspace_bytes(num_tokens, num_topk) > workspace_bytes)
        return NANOEP_ERR_WORKSPACE;
    const int window = rebuild_window_tokens(num_tokens, num_topk, hidden, knobs);
    const int64_t windows = (num_tokens + window - 1) / window;
    int sort_size = 2;
    while (sort_size < window * num_topk)
        sort_size *= 2;
    const int64_t capacity_entries = (num_tokens + kOrderTokens - 1) / kOrderTokens * kOrderTokens * num_topk;
    auto* window_counts = static_cast<int32_t*>(workspace);
    auto stream = static_cast<hipStream_t>(stream_handle);
    if (host_count != nullptr)
        __atomic_store_n(host_count, int64_t{-1}, __ATOMIC_RELEASE);
    rebuild_table_kernel<<<static_cast<unsigned>(windows), kRebuildThreads, 0, stream>>>(
        recv_metadata, dst_slots, recv_count, expanded_capacity, num_tokens, num_topk, window, token_slots, window_counts);
    NANOEP_HIP_TRY(hipGetLastError());
    rebuild_order_kernel<<<static_cast<unsigned>(windows), kRebuildThreads, static_cast<size_t>(sort_size) * 8, stream>>>(
        token_slots, window_counts, num_tokens, num_topk, window, static_cast<int>(windows), sort_size, slot_order, capacity_entries,
        host_count, host_tag);
    NANOEP_HIP_TRY(hipGetLastError());
    return NANOEP_OK;
}

int nanoep_wait_counts(int64_t* host_counts, void* stream_handle, double timeout_seconds,
                       int64_t out[NANOEP_HOST_COUNT_WORDS]) {
    if (host_counts == nullptr || out == nullptr)
        return NANOEP_ERR_INVALID_ARGUMENT;
    auto stream = static_cast<hipStream_t>(stream_handle);
    // The wait is a plain spin on the mailbox word: the counts usually arrive within microseconds,
    // and whoever waits for them wants to know at once.  The clock is read every 256 spins; the
    // stream is only asked how it is doing every 100 us of waiting (the question itself takes the
    // runtime microseconds, during which a published count would go unnoticed).
    timespec start{};
    clock_gettime(CLOCK_MONOTONIC, &start);
    double next_stream_check = 100e-6;
    uint64_t spins = 0;
    while (true) {
        const int64_t received = __atomic_load_n(&host_counts[0], __ATOMIC_ACQUIRE);
        if (received >= 0)
            break;
        if ((++spins & 0xff) == 0) {
            // the clock first: a caller with no patience left is answered without touching the stream
            timespec now{};
            clock_gettime(CLOCK_MONOTONIC, &now);
            const double elapsed = (now.tv_sec - start.tv_sec) + 1e-9 * (now.tv_nsec - start.tv_nsec);
            if (elapsed > timeout_seconds) {
                // a last look at the mailbox, and at a stream that may have failed rather than stalled
                if (__atomic_load_n(&host_counts[0], __ATOMIC_ACQUIRE) >= 0)
                    break;
                if (stream != nullptr) {
                    const hipError_t state = hipStreamQuery(stream);
                    if (state != hipSuccess && state != hipErrorNotReady) {
                        g_last_hip_error = state;
                        return NANOEP_ERR_HIP;
                    }
                }
                return NANOEP_ERR_TIMEOUT;
            }
            if (elapsed < next_stream_check)
                continue;
            next_stream_check = elapsed + 100e-6;
            // A finished (or failed) stream with no published count means the layout never ran.
            const hipError_t state = hipStreamQuery(stream);
            if (state != hipErrorNotReady) {
                if (state != hipSuccess) {
                    g_last_hip_error = state;
                    return NANOEP_ERR_HIP;
                }
                if (__atomic_load_n(&host_counts[0], __ATOMIC_ACQUIRE) >= 0)
                    break;
                return NANOEP_ERR_TIMEOUT;
            }
        }
    }
    for (int i = 0; i < NANOEP_HOST_COUNT_WORDS; ++i)
        out[i] = __atomic_load_n(&host_counts[i], __ATOMIC_RELAXED);
    return out[3] != 0 ? NANOEP_ERR_ROUTING : NANOEP_OK;
}

}  // extern "C"

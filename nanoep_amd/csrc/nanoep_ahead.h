// Source rows that a layout reads ahead for the dispatch behind it: the host's plan and the vectors every lane takes.  Nothing
// here needs a device, so that a test can walk whole grids on the host.
#ifndef NANOEP_AHEAD_H_
#define NANOEP_AHEAD_H_

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nanoep {

// Vectors a lane of the workgroups that read ahead has in flight, and what a wavefront of them reads.
constexpr int kAheadLoads = 8;
constexpr int kAheadWaveVectors = kAheadLoads * 64;

// Workgroups behind a launch's own, as many on every XCD; no workgroups: nothing is read.
struct AheadPlan {
    uint32_t blocks;
    uint32_t vectors;  // 16-byte vectors of all source rows
    uint32_t share;    // of an XCD's part of them
};

// Workgroups of `block_waves` wavefronts that read at most `bytes` in all, and no XCD more than its share.
inline AheadPlan plan_ahead(int64_t tokens, int64_t row_vectors, int64_t window_tokens, int64_t xcds, int64_t block_waves, int64_t bytes) {
    const int64_t window_rows = (tokens + window_tokens - 1) / window_tokens * window_tokens;
    if (window_rows * row_vectors >= (int64_t{1} << 31))
        return {0, 0, 0};
    AheadPlan plan{};
    plan.vectors = static_cast<uint32_t>(tokens * row_vectors);
    plan.share = static_cast<uint32_t>((window_rows + xcds - 1) / xcds * row_vectors);
    const int64_t most = (plan.share + int64_t{kAheadWaveVectors} * block_waves - 1) / (kAheadWaveVectors * block_waves);
    const int64_t allowed = bytes / (int64_t{kAheadWaveVectors} * 16) / xcds / block_waves;
    plan.blocks = static_cast<uint32_t>((most < allowed ? most : allowed) * xcds);
    return plan;
}

// Vectors [first, end) are one wavefront's: wavefront `wave` of the `ordinal`-th such workgroup on XCD `xcd`.
struct AheadRange {
    uint64_t first;
    uint64_t end;
};

__host__ __device__ inline AheadRange ahead_range(uint32_t vectors, uint32_t share, uint32_t xcd, uint32_t ordinal, uint32_t block_waves, uint32_t wave) {
    const uint64_t share_first = static_cast<uint64_t>(xcd) * share;
    const uint64_t share_end = share_first + share < vectors ? share_first + share : vectors;
    const uint64_t first = share_first + (static_cast<uint64_t>(ordinal) * block_waves + wave) * kAheadWaveVectors;
    return {first, first + kAheadWaveVectors < share_end ? first + kAheadWaveVectors : share_end};
}

// The vector a lane reads with its `load`-th load; lanes behind the end of a range that is not empty repeat its first.
__host__ __device__ inline uint64_t ahead_vector(const AheadRange& range, uint32_t load, uint32_t lane) {
    const uint64_t vector = range.first + load * 64u + lane;
    return vector < range.end ? vector : range.first;
}

// Bytes that the workgroups of a plan read (the launch's own end with workgroup `work_blocks` - 1).
inline int64_t ahead_bytes(const AheadPlan& plan, uint32_t work_blocks, uint32_t xcds, uint32_t block_waves) {
    int64_t read = 0;
    for (uint32_t block = work_blocks; block < work_blocks + plan.blocks; ++block)
        for (uint32_t wave = 0; wave < block_waves; ++wave) {
            const AheadRange range = ahead_range(plan.vectors, plan.share, block % xcds, (block - work_blocks) / xcds, block_waves, wave);
            read += range.first < range.end ? static_cast<int64_t>(range.end - range.first) * 16 : 0;
        }
    return read;
}

}  // namespace nanoep

#endif  // NANOEP_AHEAD_H_

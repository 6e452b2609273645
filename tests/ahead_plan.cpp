// The plan and the index arithmetic of nanoep_ahead.h, walked over whole grids for tests/test_ahead_plan.py.
#include "nanoep_ahead.h"

using namespace nanoep;

extern "C" {

void plan(int64_t tokens, int64_t row_vectors, int64_t window, int64_t xcds, int64_t block_waves, int64_t bytes, int64_t out[3]) {
    const AheadPlan p = plan_ahead(tokens, row_vectors, window, xcds, block_waves, bytes);
    out[0] = p.blocks, out[1] = p.vectors, out[2] = p.share;
}

int64_t bytes_of(int64_t blocks, int64_t vectors, int64_t share, int64_t work_blocks, int64_t xcds, int64_t block_waves) {
    return ahead_bytes({static_cast<uint32_t>(blocks), static_cast<uint32_t>(vectors), static_cast<uint32_t>(share)},
                       static_cast<uint32_t>(work_blocks), static_cast<uint32_t>(xcds), static_cast<uint32_t>(block_waves));
}

// Counts in reader[v] the lanes whose own vector v is (not those that repeat a range's first), and puts the XCD into xcd_of[v].
// Returns the largest vector any lane loads, -1 if none does.
int64_t walk(int64_t blocks, int64_t vectors, int64_t share, int64_t work_blocks, int64_t xcds, int64_t block_waves, uint8_t* reader,
             int8_t* xcd_of, int64_t length) {
    int64_t largest = -1;
    for (int64_t block = work_blocks; block < work_blocks + blocks; ++block)
        for (int64_t wave = 0; wave < block_waves; ++wave) {
            const uint32_t xcd = static_cast<uint32_t>(block % xcds);
            const AheadRange range = ahead_range(static_cast<uint32_t>(vectors), static_cast<uint32_t>(share), xcd,
                                                 static_cast<uint32_t>((block - work_blocks) / xcds), static_cast<uint32_t>(block_waves),
                                                 static_cast<uint32_t>(wave));
            if (range.first >= range.end)
                continue;
            for (uint32_t load = 0; load < kAheadLoads; ++load)
                for (uint32_t lane = 0; lane < 64; ++lane) {
                    const int64_t vector = static_cast<int64_t>(ahead_vector(range, load, lane));
                    largest = vector > largest ? vector : largest;
                    if (vector < length && vector == static_cast<int64_t>(range.first + load * 64 + lane)) {
                        ++reader[vector];
                        xcd_of[vector] = static_cast<int8_t>(xcd);
                    }
                }
        }
    return largest;
}
}

// How a product's feature columns are dealt out over work-groups (spmm.hip).  Host arithmetic only.
#pragma once
#include <cstdint>

namespace drone {

// Slices: the feature columns are dealt out over 2^bits work-groups per chunk or piece, each with lane groups that much
// narrower.  For one thing that halves the serial chain of a row, in a matrix so small that the GPU still holds all the
// wavefronts; us at K = 128 without / with: 4,001 vertices and 60 K entries 43 / 28, 20,003 hub-heavy ones and 0.3 M entries
// 57 / 46, epoch on 2,708 vertices 165 / 159.  With more wavefronts than that their fixed costs count: 30,001 vertices 72 / 78.
constexpr int kResidentWaves = 8192;
constexpr int kMostLanes = 64, kLeastLanes = 4;  // of a lane group, 4 columns a lane
constexpr int kMostSlices = kMostLanes / kLeastLanes;
// For another, work-groups go round the eight XCDs in turn, so an XCD always gets the same slice (of a power of two of them):
// its L2 holds that many times more feature rows, and a band has as many more columns.  Worth it with whole 128-byte lines,
// slices that are all nearly full, and an operand larger than the L2s together; us without / with: 0.25 M vertices and 6 M
// entries at K = 128 663 / 541, 1 M vertices and 16 M entries 1,811 / 1,640, the 232,965-vertex step 8,627 / 7,893, 1 M vertices
// and 32 M entries at K = 256 7,976 / 6,587; but 0.2 M vertices at K = 100 (64 + 36, or 52 + 48 across lines) 312 / 372, and
// with 32 columns a slice the step took 9,843.
constexpr int kLineFloats = 32, kSliceCols = 2 * kLineFloats;
constexpr int64_t kAllL2Bytes = 32 << 20;
inline int line_slice_bits(int K, int n_cols)
{
    const int bits = K > 2 * kSliceCols ? 2 : 1, free = (kSliceCols << bits) - K;
    return free >= 0 && free <= kSliceCols / 4 && (int64_t)n_cols * K * (int64_t)sizeof(float) > kAllL2Bytes ? bits : 0;
}

// A launch has fewer than 2^32 work-items a dimension.  Unsliced, 2^31 entries make at most 2^26 chunks (two for 65 entries), 2^24
// work-groups of 256; slices multiply that, so a matrix of many chunks has fewer of them: from 33.5 M chunks on where there were
// two, from 16.8 M where there were four.
constexpr int64_t kMostWorkItems = (1ll << 32) - 1;

struct Slicing {
    int lanes;  // of a lane group
    int bits;
};
// K >= 4 columns; waves: pieces and chunks, in `blocks` work-groups of `threads`; whole_lines: the operand's rows are 128-byte lines.
inline Slicing slicing(int K, int n_cols, bool whole_lines, int64_t waves, int64_t blocks, int threads)
{
    Slicing s{kLeastLanes, line_slice_bits(K, n_cols)};
    while (s.lanes < kMostLanes && s.lanes * 4 < K) s.lanes *= 2;  // the smallest lane group that covers K, or a slice of it
    if (s.bits > 0 && whole_lines) {
        s.lanes = kSliceCols / 4;
        for (; s.bits > 0 && (blocks << s.bits) * threads > kMostWorkItems; --s.bits) s.lanes *= 2;
        return s;
    }
    for (s.bits = 0; s.lanes > kLeastLanes && 2 * waves <= kResidentWaves; waves *= 2) {
        ++s.bits;
        s.lanes /= 2;
    }
    return s;
}

}  // namespace drone

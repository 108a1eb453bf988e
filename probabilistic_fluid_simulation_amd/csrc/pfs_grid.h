// Launch sizes for item counts up to 2^31 - 1.  Plain C++: no HIP here.
#pragma once

namespace pfs {

// Blocks of `per` items for n of them.
constexpr int blocks_for(long long n, int per) { return (int)((n + per - 1) / per); }

// A grid's two dimensions for that many blocks of 256 threads: one dimension
// takes less than 2^32 threads, so rows of 2^23 blocks.
struct Blocks {
    unsigned x, y;
};
constexpr Blocks block_rows(int blocks) {
    constexpr int kRow = 1 << 23;
    return blocks <= kRow ? Blocks{(unsigned)blocks, 1u}
                          : Blocks{(unsigned)kRow, (unsigned)blocks_for(blocks, kRow)};
}

}  // namespace pfs

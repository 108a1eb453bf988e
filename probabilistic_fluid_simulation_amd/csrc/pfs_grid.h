// Launch sizes for item counts up to 2^31 - 1.  Plain C++: no HIP here.
#pragma once

namespace pfs {

// Blocks of `per` items for n of them.
constexpr int blocks_for(long long n, int per) { return (int)((n + per - 1) / per); }

}  // namespace pfs

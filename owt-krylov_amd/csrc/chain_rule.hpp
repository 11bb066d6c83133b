// When the triangular sweeps may run as chains (k_tri_rows16).  Host code
// without device headers.
#pragma once

#include <algorithm>
#include <cstdint>

namespace owtk {

// Entries of one row in one direction: the widest slot count that is built.
constexpr int kChainEntries = 16;

// Rows of one block: the largest that the sweeps are tested with.  It is no
// limit of the kernel, which keeps 53 KB of LDS whatever the block and numbers
// far rows in 16 bits, nor a crossover: ILU(0) applies over 524,288
// Hilbert-ordered vertices, block 3, level sets / chains in us: 4,431 / 131 in
// blocks of 4,096 rows, 8,390 / 256 of 8,192, 16,805 / 508 of 16,384, and
// 46,413 / 1,024 of 32,767.
constexpr std::int64_t kChainRows = 16384;

// Rows past a chain's end that a wave's loads and addresses run on by: the
// chunks of its longest chain are rounded up to the look-ahead P <= 4, and the
// preparing wave is P + 1 chunks of 16 rows ahead.
constexpr std::int64_t kChainOverrun = 256;

// The chains' byte offsets are 32-bit: from the first row of a wave's first
// block over all rows of the blocks that its four chains, one per (block,
// component), lie in, in 8-byte vectors of bs components.
inline bool chain_offsets_fit(std::int64_t blocks, std::int64_t max_block_rows, std::int64_t bs)
{
    // (a wave's first chain is a multiple of four)
    const std::int64_t spanned = std::min<std::int64_t>(blocks, bs == 1 ? 4 : 2);
    return (spanned * max_block_rows + kChainOverrun) * bs <= 0x7fffffff / 8;
}

} // namespace owtk

"""The rule that keeps the chain sweeps' 32-bit byte offsets in range, against every offset the kernel forms."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "owt-krylov_amd" / "csrc"

# For every workgroup: the offsets of its four chains' rows from the first row of the first chain's block, the steps
# past the longest chain's end (chunks rounded up to four, loads five chunks ahead) and the backward sweep's steps
# before the start.  Prints the extremes in 64 bits and the rule's answer.
PROGRAM = r"""
#include "chain_rule.hpp"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv)
{
    const std::int64_t rows = std::atoll(argv[1]), block = std::atoll(argv[2]), bs = std::atoll(argv[3]);
    const std::int64_t blocks = (rows + block - 1) / block, chains = blocks * bs, row_bytes = 8 * bs;
    const std::int64_t longest = rows < block ? rows : block;
    auto count = [&](std::int64_t b) { return b + 1 < blocks ? block : rows - b * block; };
    std::int64_t high = 0, low = 0;
    for (std::int64_t first = 0; first < chains; first += 4) {
        std::int64_t chunks = 0;
        for (std::int64_t k = 0; k < 4; ++k) {
            const std::int64_t chain = std::min(first + k, chains - 1), n = count(chain / bs);
            chunks = std::max(chunks, (n + 15) / 16);
        }
        chunks = (chunks + 3) / 4 * 4;
        for (std::int64_t k = 0; k < 4; ++k) {
            const std::int64_t chain = std::min(first + k, chains - 1), b = chain / bs, c = chain % bs;
            const std::int64_t at = (b - first / bs) * block * row_bytes + 8 * c;
            const std::int64_t last = at + (count(b) - 1) * row_bytes;
            high = std::max(high, std::max(last, at + ((chunks + 5) * 16 + 15) * row_bytes));
            low = std::min(low, last - ((chunks + 5) * 16 + 15) * row_bytes);
        }
    }
    std::printf("%lld %lld %d\n", (long long)high, (long long)low, owtk::chain_offsets_fit(blocks, longest, bs) ? 1 : 0);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rule")
    (folder / "rule.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", "-O2", "-I", str(CSRC), str(folder / "rule.cpp"), "-o", str(folder / "rule")],
                   check=True)
    return folder / "rule"


@pytest.mark.parametrize("rows,block,bs,fits", [
    (1, 1, 1, True), (2_097_152, 4096, 3, True), (1024, 1024, 1296, True), (100_000, 16384, 1, True),
    (16384, 16384, 16_000, True), (16384, 16384, 16_384, False), (40_000, 16384, 8_000, True),
    (40_000, 16384, 8_200, False), (512, 512, 349_525, True), (512, 512, 524_289, False), (20, 1, 1_000_001, True),
    (20, 1, 1_100_000, False)])
def test_offsets_stay_in_range_where_the_rule_says_so(program, rows, block, bs, fits):
    out = subprocess.run([program, str(rows), str(block), str(bs)], check=True, capture_output=True, text=True)
    high, low, answer = map(int, out.stdout.split())
    assert answer == fits
    if fits:
        assert high < 2 ** 31 and low >= -(2 ** 31)

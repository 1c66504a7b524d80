"""The work items of the split product (split_items.hpp, compiled here for the host): every pair of a row block and
a column at or below its diagonal block belongs to exactly one item, longest items first; and the dimensions at
which test_gpu_split_layouts.py checks the product have layouts of several blocks a chunk."""
import subprocess

import numpy as np
import pytest
from conftest import ROOT

ROWS = 256
SOURCE = """
#include <cstdio>
#include "split_items.hpp"
int main() {
    long long N;
    while (std::scanf("%lld", &N) == 1) {
        const auto l = xatu_dev::split_layout(N, 256, 2.0 * 256 * 32 * 8);
        std::printf("%lld", static_cast<long long>(l.chunk));
        for (const auto& i : l.items) std::printf(" %d %d %lld", i.block, i.chunk, static_cast<long long>(i.columns));
        std::printf("\\n");
    }
}
"""


@pytest.fixture(scope="module")
def layout(tmp_path_factory):
    d = tmp_path_factory.mktemp("items")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT / 'xatu_amd' / 'csrc' / 'device'}", str(d / "main.cpp"), "-o",
                    str(d / "main")], check=True)

    def run(N):
        out = subprocess.run([str(d / "main")], input=str(N), capture_output=True, text=True, check=True).stdout.split()
        return int(out[0]), np.array(out[1:], dtype=np.int64).reshape(-1, 3)
    return run


@pytest.mark.parametrize("N", [2, 254, 256, 258, 1000, 2304, 5184, 5892, 7000, 8978, 9216, 9248, 9604, 12996, 14400, 20736,
                               36864, 50000, 70002])
def test_every_block_once(layout, N):
    chunk, items = layout(N)
    blocks = -(-N // ROWS)
    assert chunk % ROWS == 0 and np.all(np.diff(items[:, 2]) <= 0)
    seen = np.zeros((blocks, blocks), dtype=int)  # row block, column block
    for b, c, columns in items:
        first, end = max(b * ROWS, c * chunk), min(N, (c + 1) * chunk)
        assert columns == end - first > 0
        seen[b, first // ROWS:-(-end // ROWS)] += 1
    assert np.array_equal(seen, np.triu(np.ones((blocks, blocks), dtype=int)))


@pytest.mark.parametrize("N,blocks", [(9216, 3), (9604, 3), (12996, 6), (8978, 3), (9248, 3)])
def test_layouts_of_the_product_tests(layout, N, blocks):
    assert layout(N)[0] == blocks * ROWS

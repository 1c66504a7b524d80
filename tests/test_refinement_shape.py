"""The block and basis of a mixed solve's FP64 refinement (refinement.hpp, compiled here for the host): whenever
the states wanted fit the device Rayleigh-Ritz kernel, so do block and basis, whatever the guard vectors ask for."""
import subprocess

import pytest
from conftest import ROOT

SOURCE = """
#include <cstdio>
#include "refinement.hpp"
int main() {
    long long N; int nev, b, resident, rows;
    while (std::scanf("%lld %d %d %d %d", &N, &nev, &b, &resident, &rows) == 5) {
        const auto s = xatu_dev::refinement_shape(N, nev, b, resident, rows, 32, 128);
        std::printf("%d %d\\n", s.block, s.basis);
    }
}
"""


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    d = tmp_path_factory.mktemp("refinement")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT / 'xatu_amd' / 'csrc' / 'device'}", str(d / "main.cpp"), "-o",
                    str(d / "main")], check=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]
    return run


def test_fits_the_device_kernel(shape):
    cases = [(N, nev, b, resident, rows) for nev in range(1, 65) for b in {nev, nev + 1, max(2 * nev, 8)}
             for N in (b, b + 1, 5 * b, 36864) for resident, rows in ((0, 0), (1, 0), (0, 1))]
    for (N, nev, b, resident, rows), (block, basis) in zip(cases, shape(cases)):
        assert nev <= block <= b and basis <= N and (basis > block or basis == N)
        if nev <= 32:
            assert block <= 32 and basis <= 128, (nev, b, block, basis)
        if not resident and not rows:
            assert block == nev  # no guard vectors on the slower products
        if nev <= 26 and rows:
            assert block == min(b, nev + max(2, nev // 4))
        if resident:
            assert block <= -(-nev // 16) * 16  # whole tiles of 16 vectors

// Block and basis of the FP64 refinement of a mixed solve (host code without a device header).
#pragma once
#include <algorithm>
#include <cstdint>

namespace xatu_dev {

struct RefinementShape {
    int block, basis;
};

// nev states wanted of the N, block b of the FP32 phase; resident: the product is the resident FP64
// matrix; rows: it is the convolution on the row and column transforms; most_block, most_basis: what the
// device Rayleigh-Ritz kernel takes.
//
// Block: nev and some guard vectors, because the highest state wanted converges with its distance from the
// first state outside the block, which may be next to nothing (a block of nev took 64 iterations, 99 ms, where
// two guard vectors took 14, 47 ms: N = 36864, nev = 16; the whole FP32 block, twice nev, 53 ms). max(2, nev / 4)
// against none, N = 1875 to 36864, nev = 2 to 16, several spectra each: 0.38 to 1.05 of the time. None where the
// product recomputes tiles or takes the slower transforms over the whole mesh (sides without a factor pair),
// which cost up to 1.4 with them when the spectrum has its gap (142 x 142, nev = 5: 44 -> 63 ms). A resident FP64
// matrix is multiplied by whole tiles of 16 vectors: the guard fills the last one and does not begin another
// (four guard vectors at nev = 16, N = 2500 to 36864, four spectra each: 0.42 to 1.12 of the time, longer in
// half of them; three at nev = 15 instead of one 0.94 to 1.21). Never so many that a block which fits the device
// Rayleigh-Ritz kernel no longer does: past it an iteration waits for the host three times (nev = 27 to 32, N =
// 2500 and 9216, two spectra each: 1.02 to 1.39 times as long with all the guard vectors).
// Basis: 6 blocks up to that kernel's limit (4 blocks: up to 1.2 of the time).
inline RefinementShape refinement_shape(int64_t N, int nev, int b, bool resident, bool rows, int most_block,
                                        int most_basis) {
    const int guard = resident || rows ? std::max(2, nev / 4) : 0;
    RefinementShape s;
    s.block = std::min({b, nev + guard, resident ? (nev + 15) / 16 * 16 : b});
    if (nev <= most_block) s.block = std::min(s.block, most_block);
    s.basis = static_cast<int>(
        std::min<int64_t>(N, std::max({4 * s.block, std::min(6 * s.block, most_basis), s.block + 1})));
    return s;
}

}  // namespace xatu_dev

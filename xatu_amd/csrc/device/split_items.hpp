// Work items of the split product (host code without a device header): pairs (row block b, column chunk c) of
// the chunks at or below b's diagonal block, the longest item first.
#pragma once
#include <algorithm>
#include <cstdint>
#include <functional>
#include <queue>
#include <vector>

namespace xatu_dev {

struct SplitItem {
    int block, chunk;
    int64_t columns;  // of the chunk, from the diagonal block on
};
struct SplitLayout {
    int64_t chunk = 0;  // columns per chunk, a multiple of the row block
    std::vector<SplitItem> items;
};

// The layout of a matrix of dimension N with row blocks of `rows`; partial: bytes of direct partial sums
// that an item writes and the reduction reads back. The chunk is the multiple of the row block with the shortest
// schedule of its items on the CUs (one workgroup each; about 22 us per 256 x 256 block and 8 us to start and end
// an item, measured at N up to 14400; at N = 36864, which HBM bounds, the estimate says 1.03 ms where the product
// takes 1.35 to 1.57) plus the partial sums: at small N short chunks, so that every CU has work (a fixed 4096
// left 84 items, the longest 16 blocks, at N = 9216), at N = 36864 chunks of 1536. Products with staging and
// reduction, 4096 -> now: N = 2304 217 -> 58 us, 5184 361 -> 67, 9216 387 -> 136, 14400 414 -> 280, 20736 517 -> 517,
// 36864 1572 -> 1571.
inline SplitLayout split_layout(int64_t N, int64_t rows, double partial) {
    const int64_t B = (N + rows - 1) / rows;
    constexpr int kCus = 256, kMaxItems = 2048;
    SplitLayout best;
    double best_us = 1e300;
    for (int blocks : {1, 2, 3, 4, 6, 8, 12, 16}) {
        const int64_t chunk = static_cast<int64_t>(blocks) * rows;
        // skip layouts of far more items than CUs while a longer chunk remains
        if (blocks < 16 && B * B / (2 * blocks) > kMaxItems) continue;
        std::vector<SplitItem> it;
        for (int64_t ch = 0; ch * chunk < N; ++ch)
            for (int64_t b = 0; b < B; ++b) {
                const int64_t rb0 = b * rows, cb = ch * chunk;
                if (rb0 >= cb + chunk) continue;
                it.push_back({static_cast<int>(b), static_cast<int>(ch), std::min(N, cb + chunk) - std::max(rb0, cb)});
            }
        std::stable_sort(it.begin(), it.end(), [](const SplitItem& x, const SplitItem& y) { return x.columns > y.columns; });
        std::priority_queue<double, std::vector<double>, std::greater<double>> cu(std::greater<double>(),
                                                                                 std::vector<double>(kCus, 0.0));
        double last = 0.0;
        for (const SplitItem& i : it) {
            const double t = cu.top() + 8.0 + 22.0 * static_cast<double>(i.columns) / rows;
            cu.pop();
            cu.push(t);
            last = std::max(last, t);
        }
        // microseconds for the partial sums, written and read
        const double us = last + it.size() * partial / 5e6;
        if (us < best_us) {
            best_us = us;
            best.items.swap(it);
            best.chunk = chunk;
        }
    }
    return best;
}

}  // namespace xatu_dev

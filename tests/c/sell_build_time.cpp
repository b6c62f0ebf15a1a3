// Time of a small SELL copy in ranges of 64 rows and of 2048 (microseconds, the
// least of many builds each): prints the two.
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <vector>

#include "tiled_layout.h"

using npbcg_detail::SellBlocks;

int main() {
    const int n = 500, per = 60;
    std::vector<int> rowstr(n + 1, 0), colidx;
    for (int j = 0; j < n; j++) {
        for (int k = 0; k < per; k++) colidx.push_back(k * 8 + j % 8);
        rowstr[j + 1] = (int)colidx.size();
    }
    const std::vector<double> a(colidx.size(), 1.0);
    double best[2] = {1e30, 1e30};
    for (int run = 0; run < 40; run++)
        for (int i = 0; i < 2; i++) {
            SellBlocks<float> m;
            const auto t0 = std::chrono::steady_clock::now();
            if (!npbcg_detail::build_sell_blocks(n, rowstr.data(), colidx.data(), a.data(), 20000,
                                                 i == 0 ? 64 : 2048, &m))
                return 1;
            const std::chrono::duration<double, std::micro> d =
                std::chrono::steady_clock::now() - t0;
            best[i] = std::min(best[i], d.count());
        }
    std::printf("%.1f %.1f\n", best[0], best[1]);
    return 0;
}

// lq::decode_split: every task of every chunk is taken by exactly one
// workgroup, and the longest CU works at most one round longer than when the
// batch is cut into equal runs of whole rounds, over batches of 1 .. 2000 chunks.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "lq_launch.h"

using lq::DecodeSplit;

// rounds of 16 tasks on the longest CU; a chunk's LUTs count as one more.
// taken (nullable): per (chunk, task) the workgroups that take it
static int64_t longest(const DecodeSplit& d, int64_t n_chunks, int64_t per_chunk, int64_t cus, std::vector<int>* taken) {
    std::vector<int64_t> busy(cus, 0);
    for (int64_t wg = 0; wg < d.grid; wg++) {
        const int64_t wc = d.wpc > 0 ? wg / d.wpc : 0;
        const int64_t first = wc * d.span + (wg - wc * d.wpc) * d.tpw;
        const int64_t lim = d.wpc > 0 ? (wc + 1) * d.span : n_chunks * d.span;
        const int64_t last = std::min(first + d.tpw, lim);
        int64_t cost = 0;
        for (int64_t t = first; t < last;) {
            const int64_t chunk = t / d.span, tend = std::min((chunk + 1) * d.span, last);
            const int64_t end = std::min(tend, chunk * d.span + per_chunk);
            cost += 1 + (std::max<int64_t>(end - t, 0) + 15) / 16;
            if (taken)
                for (int64_t k = t; k < end; k++) (*taken)[chunk * per_chunk + k - chunk * d.span]++;
            t = tend;
        }
        *std::min_element(busy.begin(), busy.end()) += cost;   // the next free CU takes it
    }
    return *std::max_element(busy.begin(), busy.end());
}

int main() {
    int64_t checked = 0, bad = 0;
    const int64_t sizes[] = {1, 2, 5, 15, 16, 17, 33, 64, 100, 512};
    for (int64_t cus : {256, 64})
        for (int64_t n = 1; n <= 2000; n = n < 600 ? n + 1 : n + 61)
            for (int64_t per : sizes) {
                if (n * per > 200000) continue;
                const DecodeSplit d = lq::decode_split(n, per, cus);
                std::vector<int> taken(n * per, 0);
                const int64_t got = longest(d, n, per, cus, &taken);
                const int64_t rounds = (per + 15) / 16, run = (n * rounds + cus - 1) / cus;
                const int64_t even = longest({16 * rounds, 16 * run, 0, (n * rounds + run - 1) / run}, n, per, cus, nullptr);
                const bool ok = got <= even + 1 && d.grid > 0 && d.grid <= std::max(n, cus) &&
                                std::all_of(taken.begin(), taken.end(), [](int c) { return c == 1; });
                checked++;
                if (!ok && bad++ < 10)
                    printf("n=%lld per=%lld cus=%lld: %lld rounds, runs of whole rounds %lld\n", (long long)n, (long long)per,
                           (long long)cus, (long long)got, (long long)even);
            }
    printf("%lld batches, %lld bad\n", (long long)checked, (long long)bad);
    return bad != 0;
}

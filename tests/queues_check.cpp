// Host-only check of the order of a batch's tiles (uvt_queues.hpp; built and
// run by tests/test_queues_host.py, no GPU).  The persistent kernel's drawing
// is run here for launches of one to several thousand workgroups, in turns and
// one workgroup after another: every tile is run once, by a draw inside the
// list, every workgroup ends after at most two failed draws, every queue that
// holds tiles has a workgroup that draws from it, and the shared queue goes
// most work first.
#include <stdio.h>

#include "uvt_queues.hpp"

using namespace uvt;

static int fails = 0;
#define CHECK(c, ...)                                          \
    do {                                                       \
        if (!(c) && ++fails <= 10) {                           \
            fprintf(stderr, "line %d: %s: ", __LINE__, #c);    \
            fprintf(stderr, __VA_ARGS__);                      \
            fprintf(stderr, "\n");                             \
        }                                                      \
    } while (0)

static int64_t work(const BatchTile& t) { return (int64_t)(t.k_hi - t.k_lo) * (t.cfg ? 64 * 64 : 128 * 128); }

// Problems of rows x cols tiles each.
static std::vector<BatchTile> batch(const std::vector<std::pair<int, int>>& probs)
{
    std::vector<BatchTile> v;
    for (int p = 0; p < (int)probs.size(); ++p)
        for (int r = 0; r < probs[p].first; ++r)
            for (int c = 0; c < probs[p].second; ++c)
                v.push_back(BatchTile{p, r * 128, 128, c * 128, 0, r * 128 + 128, p % 3 == 1});
    return v;
}

static void run(const std::vector<std::pair<int, int>>& probs, int grid)
{
    std::vector<BatchTile> v = batch(probs);
    const int all = (int)v.size();
    const TileQueues q = deal_tiles(v, grid, work);
    const int launched = grid < all ? grid : all;
    CHECK((int)v.size() == all && q.first[kQueues + 1] == all && q.first[0] == launched, "%d of %d", (int)v.size(), all);
    std::vector<std::vector<char>> seen(probs.size());
    for (size_t p = 0; p < probs.size(); ++p) seen[p].assign(probs[p].first * probs[p].second, 0);
    for (const BatchTile& t : v) seen[t.prob][t.r0 / 128 * probs[t.prob].second + t.c0 / 128]++;
    for (auto& s : seen)
        for (char c : s) CHECK(c == 1, "tile listed %d times", c);
    for (int j = 0; j < kQueues; ++j)
        CHECK(q.first[j] <= q.first[j + 1] && (q.first[j] == q.first[j + 1] || j < launched), "queue %d", j);
    for (int i = q.first[kQueues] + 1; i < all; ++i) CHECK(work(v[i - 1]) >= work(v[i]), "tile %d", i);
    for (int turns = 0; turns < 2; ++turns) {
        std::vector<int> ran(all, 0), counter(kQueues + 1, 0), failed(launched, 0);
        std::vector<char> own(launched), done(launched, 0);
        auto draw = [&](int b) {  // as k_batch_f64
            const int x = b % kQueues, size = q.first[x + 1] - q.first[x];
            const int shared = q.first[kQueues], rest = q.first[kQueues + 1] - shared;
            int t = -1;
            if (size == 0 && rest == 0) return -1;
            if (own[b]) {
                const int i = counter[x]++;
                if (i < size) t = q.first[x] + i;
                else ++failed[b];
            }
            if (t < 0 && rest > 0) {
                const int i = counter[kQueues]++;
                if (i < rest) t = shared + i;
                else ++failed[b];
            }
            own[b] = t < shared;
            return t;
        };
        for (int b = 0; b < launched; ++b) {
            ran[b]++;
            own[b] = q.first[b % kQueues + 1] > q.first[b % kQueues];
        }
        for (int left = launched; left > 0;)
            for (int b = 0; b < launched; ++b) {
                while (!done[b]) {
                    const int t = draw(b);
                    if (t < 0) {
                        done[b] = 1;
                        --left;
                    } else {
                        CHECK(t < all, "tile %d", t);
                        if (t < all) ran[t]++;
                    }
                    if (turns == 0) break;
                }
            }
        for (int t = 0; t < all; ++t) CHECK(ran[t] == 1, "tile %d of %d run %d times, grid %d", t, all, ran[t], grid);
        for (int f : failed) CHECK(f <= 2, "%d failed draws", f);
    }
}

int main()
{
    const std::vector<std::vector<std::pair<int, int>>> cases = {
        {{1, 1}},
        {{1, 1}, {1, 1}, {1, 1}, {1, 1}, {1, 1}, {1, 1}, {1, 1}},
        std::vector<std::pair<int, int>>(9, {1, 1}),
        {{40, 30}},
        std::vector<std::pair<int, int>>(60, {32, 1}),
        std::vector<std::pair<int, int>>(60, {5, 5}),
        std::vector<std::pair<int, int>>(1200, {1, 1}),
        {{32, 8}, {1, 1}, {2, 3}, {16, 1}, {7, 2}, {32, 1}, {3, 8}, {20, 5}},
        std::vector<std::pair<int, int>>(60, {16, 8}),
    };
    for (const auto& c : cases)
        for (int grid : {1, 3, 7, 8, 9, 64, 511, 512, 5000}) run(c, grid);
    if (fails) fprintf(stderr, "%d checks failed\n", fails);
    else printf("ok\n");
    return fails != 0;
}

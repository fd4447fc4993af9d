// uvt_queues.hpp -- the order in which the persistent batch kernel runs its
// tiles (host; the kernel is k_batch_f64 in uvt_batch.hip).
//
// The tile list starts with the first tile of every workgroup (workgroup b
// runs tile b, without drawing it), then one queue per XCD (workgroup b runs
// on XCD b % 8 and draws from that queue), then one queue that all share.
// Tiles of a group, which read the same operands, run side by side on one XCD
// and find each other's panels in its L2; the shared queue, most work first,
// evens out what the XCDs' queues leave.  A workgroup ends after at most two
// failed draws.  (Drawing from the fullest other queue instead took up to
// eight counter reads and a draw per attempt, by every workgroup at once at
// the end: 200 problems of 200 x 200 90 us, now 80; 256 of 128 x 16 25.7, now
// 20.4; 512 uneven ones, n to 4096, m to 1024, 5.11 and 5.13 ms.)
#pragma once

#include <stdint.h>

#include <algorithm>
#include <vector>

namespace uvt {

struct BatchTile {
    int32_t prob, r0, rows, c0, k_lo, k_hi, cfg;  // cfg: UVT_CFG_* tile shape
};

// Queue q, kXcds of them and the shared one, holds tiles first[q] to
// first[q + 1] of the list, handed out by counter q * kCounterPad (each
// counter has a cache line of its own: side by side in one line, the draws of
// all XCDs made short batches 20-30 % slower).
constexpr int kQueues = 8, kCounterPad = 16;
struct TileQueues {
    int32_t first[kQueues + 2];
};

// Puts the tiles (in problem order) in that order for a launch of `grid`
// workgroups (fewer if there are fewer tiles); work(tile): what it costs.
//
// A queue takes groups, each a whole problem or as many of its row blocks,
// deepest first, as make up 1/64 of the batch's work; the deepest group goes
// first, to the queue with the least work so far.  Measured on 512 uneven
// problems, n to 4096, m to 1024: groups of one row block 8.97-9.00 ms, of 256
// rows 8.81-8.85, 512 8.65-8.69, 1024 8.59, whole problems 8.34-8.35; 60
// problems of 2048 x 1024, where whole problems leave the queues uneven:
// 4.27-4.30 ms by 1/32 of the work, 4.11-4.12 by 1/64, 4.14 by 1/128, 4.16 by
// 1/256.  Row blocks of a problem with one column tile share only B, and go
// singly: 60 problems of 4096 x 32 843 -> 787 us.
//
// The shared queue takes the last 128 tiles of every queue (two for each of
// its XCD's 64 workgroups), or as many as make up 1/16 of its work: 1/32 and
// 1/8 of it measured within 1 %.
template <class Work>
TileQueues deal_tiles(std::vector<BatchTile>& v, int grid, Work&& work)
{
    constexpr int kGroups = 64, kShare = 16;
    constexpr size_t kTail = 128;
    struct Group {
        size_t lo, hi;
        int64_t top, sum;  // work of its largest tile and of all of them
    };
    int64_t total = 0;
    for (const BatchTile& t : v) total += work(t);
    std::vector<Group> groups;
    for (size_t i = 0; i < v.size();) {
        size_t e = i;
        while (e < v.size() && v[e].prob == v[i].prob) ++e;
        std::stable_sort(v.begin() + i, v.begin() + e,
                         [](const BatchTile& a, const BatchTile& b) { return a.r0 > b.r0; });
        const bool wide = i + 1 < e && v[i].r0 == v[i + 1].r0;
        while (i < e) {
            Group g{i, i, 0, 0};
            do {  // one row block
                for (const int r0 = v[g.hi].r0; g.hi < e && v[g.hi].r0 == r0; ++g.hi) {
                    g.top = std::max(g.top, work(v[g.hi]));
                    g.sum += work(v[g.hi]);
                }
            } while (g.hi < e && g.sum < total / kGroups && wide);
            groups.push_back(g);
            i = g.hi;
        }
    }
    std::stable_sort(groups.begin(), groups.end(), [](const Group& a, const Group& b) { return a.top > b.top; });
    std::vector<BatchTile> q[kQueues], last;
    int64_t load[kQueues] = {0};
    for (const Group& g : groups) {
        const int to = (int)(std::min_element(load, load + kQueues) - load);
        load[to] += g.sum;
        q[to].insert(q[to].end(), v.begin() + g.lo, v.begin() + g.hi);
    }
    const auto more = [&](const BatchTile& a, const BatchTile& b) { return work(a) > work(b); };
    for (auto& x : q) std::stable_sort(x.end() - std::min(x.size(), kTail), x.end(), more);
    const size_t all = v.size();
    size_t at[kQueues] = {0};
    v.clear();
    for (size_t b = 0; b < all && b < (size_t)grid; ++b) {
        size_t from = b % kQueues;
        if (at[from] == q[from].size())
            for (size_t x = 0; x < kQueues; ++x)
                if (q[x].size() - at[x] > q[from].size() - at[from]) from = x;
        v.push_back(q[from][at[from]++]);
    }
    TileQueues r;
    for (int j = 0; j < kQueues; ++j) {
        size_t e = q[j].size();
        // (a queue that no workgroup draws from goes to the shared one whole)
        for (int64_t w = 0; e > at[j] && (q[j].size() - e < kTail || w < load[j] / kShare || j >= grid);) w += work(q[j][--e]);
        r.first[j] = (int32_t)v.size();
        v.insert(v.end(), q[j].begin() + at[j], q[j].begin() + e);
        last.insert(last.end(), q[j].begin() + e, q[j].end());
    }
    std::stable_sort(last.begin(), last.end(), more);
    r.first[kQueues] = (int32_t)v.size();
    v.insert(v.end(), last.begin(), last.end());
    r.first[kQueues + 1] = (int32_t)v.size();
    return r;
}

}  // namespace uvt

// Host-only check of overlap() (uvt_overlap.hpp; built and run by
// tests/test_overlap_host.py, no GPU) against the elements themselves, for
// every pair of small blocks of one buffer.
#include <stdio.h>

#include <vector>

#include "uvt_overlap.hpp"

static bool shared(int64_t d, int rp, int cp, int ldp, int rq, int cq, int ldq)
{
    std::vector<char> used(1024, 0);
    for (int i = 0; i < rp; ++i)
        for (int j = 0; j < cp; ++j) used[512 + i * ldp + j] = 1;
    for (int i = 0; i < rq; ++i)
        for (int j = 0; j < cq; ++j)
            if (used[512 + d + i * ldq + j]) return true;
    return false;
}

int main()
{
    static double buf[1024];
    int fails = 0;
    for (int ldp = 1; ldp <= 5; ++ldp)
        for (int ldq = 1; ldq <= 5; ++ldq)
            for (int cp = 1; cp <= ldp; ++cp)
                for (int cq = 1; cq <= ldq; ++cq)
                    for (int rp = 1; rp <= 3; ++rp)
                        for (int rq = 1; rq <= 3; ++rq)
                            for (int d = -24; d <= 24; ++d) {
                                const bool want = shared(d, rp, cp, ldp, rq, cq, ldq);
                                const bool got = uvt::overlap(buf + 512, rp, cp, ldp, buf + 512 + d, rq, cq, ldq);
                                if ((want && !got) || (ldp == ldq && got != want)) ++fails;
                            }
    if (fails) fprintf(stderr, "%d checks failed\n", fails);
    else printf("ok\n");
    return fails != 0;
}

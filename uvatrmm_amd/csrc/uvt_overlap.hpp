// uvt_overlap.hpp -- whether two strided matrices share an element (host).
#pragma once

#include <stdint.h>

namespace uvt {

// P: rp x cp with leading dimension ldp; Q: rq x cq with ldq; row-major
// doubles, no dimension 0.  Exact for equal leading dimensions (blocks of one
// matrix, whose address ranges interleave); for others, true whenever the
// address ranges meet.
inline bool overlap(const double* P, int64_t rp, int64_t cp, int64_t ldp, const double* Q, int64_t rq, int64_t cq,
                    int64_t ldq)
{
    const intptr_t p = (intptr_t)P, q = (intptr_t)Q;
    if (q >= p + 8 * ((rp - 1) * ldp + cp) || p >= q + 8 * ((rq - 1) * ldq + cq)) return false;
    if (ldp != ldq || (q - p) % 8 != 0) return true;
    // Q starts dr rows and dc columns into P's layout; the columns of Q past
    // the end of a row there lie one row further down.
    const int64_t d = (q - p) / 8, dr = d >= 0 ? d / ldp : -((-d + ldp - 1) / ldp), dc = d - dr * ldp;
    const auto rows_meet = [&](int64_t r) { return r < rp && r + rq > 0; };
    return (rows_meet(dr) && dc < cp) || (rows_meet(dr + 1) && dc + cq > ldp);
}

}  // namespace uvt

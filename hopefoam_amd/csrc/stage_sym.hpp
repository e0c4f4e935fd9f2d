// Sizes of the mirror-symmetric FP64 stage kernel (stage_sym.hip) and of its operator fragments (dgh_api.cpp).
#pragma once
#include "dg_common.hpp"

namespace dg {

// The reference triangle, its nodes, its cubature rule and its face rules are symmetric under r <-> s.  Nodes
// (points) come as mirror pairs and as fixed ones on the axis; a "row" is a pair or a fixed node (point), pairs
// first.  Values at a pair enter the contractions as their sum and difference, and the sums and differences do not
// mix.
// Order 1 takes the whole operators instead: every node and point is a row of its own and there are no pairs.  Its three
// nodes fill one tile either way, and the halves need 14 products per variable and four fluxes per lane where the whole
// operators need 10 and three.
template <int N>
struct SymDims {
    static constexpr bool whole = N == 1;
    static constexpr int Np = (N + 1) * (N + 2) / 2;
    static constexpr int nfix = whole ? Np : N / 2 + 1, npair = (Np - nfix) / 2, nrow = npair + nfix;
    static constexpr int Nq = kNq[N];
    static constexpr int kFix[kMaxN + 1] = {0, Nq, 5, 6, 6, 7, 7, 10, 11};   // cubature points on the axis (1: all)
    static constexpr int qfix = kFix[N], qpair = (Nq - qfix) / 2, qrow = qpair + qfix;
    static constexpr int KE = (nrow + 3) / 4, KO = (npair + 3) / 4;     // K steps of the interpolation
    static constexpr int ME = (nrow + 15) / 16, MO = (npair + 15) / 16; // row tiles of the projection
    static constexpr int TE = (qrow + 15) / 16, TO = (qpair + 15) / 16; // point-row tiles
    static constexpr int KP = (qpair + 3) / 4, KT = (qrow + 3) / 4;     // point steps (4 point rows): with pairs, all
    static constexpr int Nfp = N + 1, Nfq = N + 2, SF = (Nfq + 3) / 4;  // K steps per face
    // fragments, 64 lanes each: interpolation of sums [TE][KE] and differences [TO][KO]; projection per point step
    // [point, mirror point][ME sums, MO differences] (steps of fixed points: the point only); lift per K step of
    // faces 0 and 2 (sums, differences) and of face 1 [ME, MO].  Whole operators: projection per point step [Pr, Ps][ME],
    // lift per K step of faces 0, 2 and 1 [ME]
    static constexpr int nV = (TE * KE + TO * KO) * 64;
    static constexpr int nP = whole ? 2 * KT * ME * 64 : (KT + KP) * (ME + MO) * 64;
    static constexpr int nL = (whole ? 3 * ME : 2 * (ME + MO)) * SF * 64;
    static constexpr int nF = nV + nP + nL;
};

}  // namespace dg

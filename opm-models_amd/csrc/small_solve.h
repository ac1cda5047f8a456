// small_solve.h -- BiCGStab with natural-order block ILU(0) on a system whose
// preconditioned vector fits in one CU's LDS (small_solve.hip).
#pragma once

#include "omodels_internal.h"

namespace omodels {

// The most scalar rows: 128 KB of doubles in LDS.  Where the other path is a
// launch per level, one workgroup is the faster one up to that limit, least so
// on cubes, which have the fewest levels.  A solve in ms, against the launches
// (and their graph replay):
//   3x3 FP32, 17x17x18 2.8 (8.4, 6.1), 43x127x1 53 (419, 216), 5461x1x1 2.8 (126, 56);
//   3x3 FP64 with wells, 16x16x16 4.0 (7.0, 6.0), 17x17x18 4.9 (8.3, 8.1);
//   2x2, lens runs of 128x64 109 (939, 487), of 4096x2 2507 (23487, 13588).
constexpr long kSmallEntries = 16384;
// And where the tile sweeps are there instead: one CU reads a system's
// matrices at some 20-40 GB/s here, so its iteration grows with the rows
// (56 us at 480 rows of 3x3 blocks in FP64, 104 at 1200, 182 at 2352), while
// the tiles' hardly does (118 us, 137, 175).  At the line, a solve in ms
// against the tiles, FP64 / FP32 inner: 16x12x8 1.26 / 1.12 (1.64 / 1.80),
// 39x39x1 15.5 / 3.6 (22.5 / 5.9), 1x1x1536 1.00 / 1.01 (1.76 / 1.92), 1536x1x1
// 1.01 / 1.02 (1.31 / 1.25); the FP32 inner solve alone would allow more rows.
constexpr long kSmallTiledEntries = 4608;
inline bool smallSystem(long rows, int bs) { return (bs == 2 || bs == 3) && rows > 0 && rows * bs <= kSmallEntries; }

// The whole solve (BiCGStabSolver::apply, bicgstabsolver.hh:120-330) in one
// launch: x, the scalars with the verdict (stop_rc -1: the iterations ran out)
// and the iteration count come back in x and ks.  w: four work vectors of
// bs * n entries.
template <class S>
void launchSmallBicgstab(int n, int bs, const LevelSchedule& L, const int* rp, const int* ci, const S* A, const S* lu,
                         const double* dinv, const S* b, S* x, S* const w[4], double tol, double absTol,
                         double maxError, int maxIter, KrylovScalars* ks, hipStream_t st);

// The factorization of such a system in one launch: lu holds the matrix and
// gets the factors (inverted pivots on the diagonal), dinv the pivots as FP64.
template <class S>
void launchSmallFactor(int n, int bs, const LevelSchedule& L, const int* rp, const int* ci, const int* diag, S* lu,
                       double* dinv, int* dFail, hipStream_t st);

}  // namespace omodels

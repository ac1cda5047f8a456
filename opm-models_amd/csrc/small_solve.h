// small_solve.h -- BiCGStab with natural-order block ILU(0) on a system whose
// preconditioned vector fits in one CU's LDS (small_solve.hip).
#pragma once

#include "omodels_internal.h"

namespace omodels {

// the most scalar rows: 128 KB of doubles in LDS
constexpr long kSmallEntries = 16384;
// and where the tile sweeps are there instead: one CU reads a system's
// matrices at some 20-40 GB/s here, so its iteration grows with the rows
// (56 us at 480 rows of 3x3 blocks, 104 at 1200, 182 at 2352), while the
// tiles' hardly does (118 us, 137, 175)
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

// krylov_device.h -- the scalar steps of BiCGStab as device functions
// (BiCGStabSolver::apply, bicgstabsolver.hh:120-330): one thread evaluates
// them on the scalars of the solve.
#pragma once

#include "omodels_internal.h"

namespace omodels {

__device__ __forceinline__ double waveMax(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
    return v;
}

__device__ __forceinline__ void markFail(KrylovScalars* ks, int tag)
{
    if (!ks->fail_code) { ks->fail_code = 2; ks->fail_tag = tag; }
}

// what the last workgroup does with the sums (s0, s1)
__device__ __forceinline__ void dotEpilogue(int mode, double s0, double s1, KrylovScalars* ks, double eps, int tagOff,
                                            double* out)
{
    if (mode == kDotValue) { *out = s0; return; }
    const int tag = ks->tag_base + tagOff;
    if (mode == kDotRho) {             // rho_i = <r0hat, r>, beta (bicgstabsolver.hh:197-206)
        ks->rho_i = s0;
        if (fabs(ks->rho) <= eps || fabs(ks->omega) <= eps) markFail(ks, tag);
        ks->beta = (s0 / ks->rho) * (ks->alpha / ks->omega);
        ks->rho = s0;
    } else if (mode == kDotAlpha) {    // denom = <r0hat, v>, alpha (:230-236)
        ks->denom = s0;
        if (fabs(s0) <= eps) markFail(ks, tag);
        ks->alpha = ks->rho / s0;
        if (fabs(ks->alpha) <= eps) markFail(ks, tag);
    } else {                           // omega = <t, s> / <t, t> (:287-292)
        if (fabs(s0) <= eps) markFail(ks, tag);
        ks->omega = s1 / s0;
        if (fabs(ks->omega) <= eps) markFail(ks, tag);
    }
}

// the test after the first half of iteration tag_base / 2 (bicgstabsolver.hh:
// 252-273) with the outcome of the previous second half (:286-318), in the
// order of the host loop; once it ends the solve, the queued kernels of
// the next iteration return at once
__device__ __forceinline__ void criterion(double mx, bool change, KrylovScalars* ks)
{
    ks->resnorm = mx;
    ks->stag_half = change ? 0 : 1;
    const int tag = ks->tag_base;
    int rc = -1, back = 0;
    if (tag > 0 && ks->fail_code && ks->fail_tag == tag - 1) { rc = 2; back = 1; }
    else if (tag > 0 && ks->stag_full_tag == tag - 1) { rc = 1; back = 1; }
    else if (ks->fail_code) rc = 2;
    else if (mx / fmax(1e-20, ks->init_norm) <= ks->tol || mx <= ks->abs_tol) rc = 0;
    else if (ks->stag_half || mx > ks->max_error) rc = 1;
    if (rc >= 0) {
        ks->stop_rc = rc;
        ks->stop_back = back;
        ks->run = 0;
    }
}

}  // namespace omodels

// small_solve.hip -- the linear solve of a small system in one workgroup.
//
// A small system is bounded by latency, not by its bytes: a natural-order
// ILU(0) sweep is a chain of levels, and with a launch per tile wave or per
// level and per vector step the chain is made of launches.  Here one workgroup
// of 8 waves keeps the preconditioned vector in LDS and runs every iteration:
// a level costs its LDS reads, some 18 dependent multiplies and adds and a
// barrier (0.21 us on narrow levels, 0.35 us with two chunks of 3x3 rows; a
// launch of one level 1.8 us and its gap), and the vector steps between the
// sweeps have no launches at all.  An FP64 iteration of 480 rows of 3x3 blocks
// 56 us (118 us by tiles), of 1536 rows of 2x2 blocks 102 us (1.2 ms by levels).
//
// Rows of a level go to the waves in chunks (16 rows of 3x3 blocks, one quad of
// lanes per row; 32 rows of 2x2 blocks, one pair), round robin over the
// waves across the levels, so that on narrow levels a wave has several levels'
// time to fetch its next two chunks: their blocks are in registers when the
// level's turn comes.  The barriers wait for LDS only; the fetches stay in flight.
//
// Per row every operation is the level-scheduled kernels' in the same order,
// and the scalar products are exact (exact_sum.h): the same bits as the solve
// by separate launches.
#include <limits>

#include "block_ops.h"
#include "krylov_device.h"
#include "small_solve.h"

namespace omodels {

namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
static_assert(LevelSchedule::kSlotPad >= 6 * kWaves, "the sweeps read the slots of chunks ahead");

// lanes per row and rows per chunk
template <int BS>
struct RowLanes {
    static constexpr int kLanes = BS == 3 ? 4 : 2, kRows = 64 / kLanes;
};

__device__ __forceinline__ void ldsBarrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// component q of the lane's row (lanes of a row: quads for BS 3, pairs for BS 2)
template <int Ctrl>
__device__ __forceinline__ float dppGet(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), Ctrl, 0xf, 0xf, true));
}
template <int Ctrl>
__device__ __forceinline__ double dppGet(double v)
{
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), Ctrl, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), Ctrl, 0xf, 0xf, true));
}
template <int BS, int Q, class T>
__device__ __forceinline__ T rowComponent(T v)
{
    if constexpr (BS == 3) return dppGet<Q * 0x55>(v);
    else return dppGet<Q == 0 ? 0xA0 : 0xF5>(v);
}

template <class S>
struct SmallArgs {
    int n, nLevels, nChunks, maxIter;
    const int4* slots;
    const int *rp, *ci;
    const S *A, *lu, *b;
    const double* dinv;
    S *x, *r, *p, *v, *t;
    KrylovScalars* ks;
    double tol, absTol, maxError;
};

// slot fields (LevelSchedule::slots)
__device__ __forceinline__ int slotLower(const int4& m) { return m.z & 0xffff; }
__device__ __forceinline__ int slotUpper(const int4& m) { return (int)((unsigned)m.z >> 16); }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// A wave's next chunk: the lane's row (component e of it), fetched ahead.
template <int BS, class S>
struct SmallChunk {
    int4 m, next;                  // this chunk's slot, and the one after the wave's other chunk
    S L[BS][BS], d;
    double D[BS];
    int c[BS];
};

// One triangular sweep: forward from d (global) into sv (LDS), backward in
// place on sv.  Every thread calls it, with sv free (forward) or complete
// (backward); on return sv is complete.  A wave holds its next two chunks; it
// passes a level's barrier before it fetches again, so the fetches' issue is
// not in the chain either.
template <int BS, class S, bool Bwd>
__device__ __forceinline__ void smallSweep(const SmallArgs<S>& a, const S* d, S* sv)
{
    constexpr int LPR = RowLanes<BS>::kLanes, RPW = RowLanes<BS>::kRows, BB = BS * BS;
    const int lane = (int)(threadIdx.x & 63u), w = uniform((int)(threadIdx.x >> 6));
    const bool row = lane % LPR < BS;
    const int e = row ? lane % LPR : 0;
    // the table has 4 kWaves empty chunks at either end
    const int4* slots = a.slots + (long)RPW * ((Bwd ? a.nChunks - 1 : 0) + LevelSchedule::kSlotPad) + lane / LPR;
    constexpr long kStep = (Bwd ? -1L : 1L) * RPW;
    auto slot = [&](int t) { return slots[t * kStep]; };
    auto levelOf = [&](const int4& m) { return uniform(Bwd ? a.nLevels - 1 - m.w : m.w); };
    auto fetch = [&](SmallChunk<BS, S>& q) {
        const int i = max(q.m.x, 0), cnt = Bwd ? slotUpper(q.m) : slotLower(q.m);
        const int k0 = Bwd ? q.m.y + slotLower(q.m) + 1 : q.m.y;
#pragma unroll
        for (int u = 0; u < BS; ++u) {
            const long k = u < cnt ? k0 + u : q.m.y;         // an entry that is there; not used
            const int c = a.ci[k];
            q.c[u] = u < cnt ? c : i;
#pragma unroll
            for (int j = 0; j < BS; ++j) q.L[u][j] = a.lu[BB * k + BS * e + j];
        }
        if (Bwd) {
#pragma unroll
            for (int j = 0; j < BS; ++j) q.D[j] = a.dinv[(long)BB * i + BS * e + j];
        } else {
            q.d = d[(long)BS * i + e];
        }
    };
    auto compute = [&](const SmallChunk<BS, S>& q) {
        if (q.m.x < 0 || !row) return;
        const int i = q.m.x, cnt = Bwd ? slotUpper(q.m) : slotLower(q.m);
        S x[BS][BS];
#pragma unroll
        for (int u = 0; u < BS; ++u)
#pragma unroll
            for (int j = 0; j < BS; ++j) x[u][j] = sv[BS * q.c[u] + j];
        S rhs = Bwd ? sv[BS * i + e] : q.d;
#pragma unroll
        for (int u = 0; u < BS; ++u) {
            S sum = q.L[u][0] * x[u][0];
#pragma unroll
            for (int j = 1; j < BS; ++j) sum += q.L[u][j] * x[u][j];
            const S next = rhs + S(-1) * sum;
            rhs = u < cnt ? next : rhs;
        }
        if (cnt > BS) {                     // rows with links beyond the grid's
            const long k0 = Bwd ? (long)q.m.y + slotLower(q.m) + 1 : (long)q.m.y;
            for (long k = k0 + BS; k < k0 + cnt; ++k) {
                const int c = a.ci[k];
                S sum = a.lu[BB * k + BS * e] * sv[BS * c];
#pragma unroll
                for (int j = 1; j < BS; ++j) sum += a.lu[BB * k + BS * e + j] * sv[BS * c + j];
                rhs += S(-1) * sum;
            }
        }
        if (Bwd) {
            double o = q.D[0] * (double)rowComponent<BS, 0>(rhs);
            o += q.D[1] * (double)rowComponent<BS, 1>(rhs);
            if constexpr (BS == 3) o += q.D[2] * (double)rowComponent<BS, 2>(rhs);
            rhs = S(0) + S(1) * (S)o;
        }
        sv[BS * i + e] = rhs;
    };
    SmallChunk<BS, S> q0, q1;
    q0.m = slot(w);
    q1.m = slot(w + kWaves);
    q0.next = slot(w + 2 * kWaves);
    q1.next = slot(w + 3 * kWaves);
    fetch(q0);
    fetch(q1);
    int l = 0, lev = levelOf(q0.m);         // l: barriers passed
    int t = w;
    auto turn = [&](SmallChunk<BS, S>& q, const SmallChunk<BS, S>& other) {
        for (; l < lev; ++l) ldsBarrier();
        compute(q);
        const int after = levelOf(other.m);
        if (after != lev) { ldsBarrier(); ++l; }
        lev = after;
        q.m = q.next;
        q.next = slot(t + 4 * kWaves);
        t += kWaves;
        fetch(q);
    };
    while (lev < a.nLevels) {
        turn(q0, q1);
        if (lev >= a.nLevels) break;
        turn(q1, q0);
    }
    for (; l < a.nLevels; ++l) ldsBarrier();
}

// out = A sv on the thread's own entries (entry k of thread t: t + 512 k)
template <int BS, class S>
__device__ __forceinline__ void smallSpmv(const SmallArgs<S>& a, const S* sv, S* out)
{
    constexpr int BB = BS * BS, U = 7;
    const int m = BS * a.n;
#pragma unroll 1
    for (int idx = (int)threadIdx.x; idx < m; idx += kThreads) {
        const int i = idx / BS, e = idx - BS * i;
        const int k1 = a.rp[i + 1];
        S acc = S(0);
#pragma unroll 1
        for (int k0 = a.rp[i]; k0 < k1; k0 += U) {
            S v[U][BS];
            int c[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u < k1 ? k0 + u : k0;
                c[u] = a.ci[k];
#pragma unroll
                for (int j = 0; j < BS; ++j) v[u][j] = a.A[(long)BB * k + BS * e + j];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                S sum = v[u][0] * sv[BS * c[u]];
#pragma unroll
                for (int j = 1; j < BS; ++j) sum += v[u][j] * sv[BS * c[u] + j];
                const S next = acc + sum;
                acc = k0 + u < k1 ? next : acc;
            }
        }
        out[idx] = acc;
    }
}

struct SmallShared {
    unsigned long long acc[2 * kAccLimbs];      // clear between products
    long long digits[2 * kAccLimbs];
    unsigned flags;                             // 3 bits a sum, clear between products
    double sum[2], wmax[kWaves];
    unsigned wany[kWaves];
    KrylovScalars ks;
};

// the sums of a.b (and with NACC = 2 of a.a, a.b) over the threads' own
// entries; thread 0 evaluates the scalars.  A barrier on either side.
template <class S, int NACC>
__device__ __forceinline__ void smallDot(int m, const S* x, const S* y, SmallShared& sh, int mode, double eps,
                                         int tagOff)
{
    constexpr int U = 4;
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    unsigned fl0 = 0u, fl1 = 0u;
#pragma unroll 1
    for (int base = (int)threadIdx.x - lane; base < m; base += U * kThreads) {      // uniform in a wave
        double v0[U], v1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = base + lane + u * kThreads;
            v0[u] = v1[u] = 0.0;
            if (idx < m) {
                const double xi = (double)x[idx];
                v0[u] = xi * (NACC == 2 ? xi : (double)y[idx]);
                if (NACC == 2) v1[u] = xi * (double)y[idx];
            }
        }
        accumulateBands<U>(v0, sh.acc, fl0);
        if (NACC == 2) accumulateBands<U>(v1, sh.acc + kAccLimbs, fl1);
    }
    if (fl0 | fl1) atomicOr(&sh.flags, fl0 | (fl1 << 3));
    __syncthreads();
    if (w < NACC) {
        unsigned long long* acc = sh.acc + w * kAccLimbs;
        const unsigned long long v0 = acc[lane], v1 = lane + 64 < kAccLimbs ? acc[lane + 64] : 0ull;
        acc[lane] = 0ull;
        if (lane + 64 < kAccLimbs) acc[lane + 64] = 0ull;
        const double s = roundLimbs(v0, v1, (sh.flags >> (3 * w)) & 7u, sh.digits + w * kAccLimbs);
        if (lane == 0) sh.sum[w] = s;
    }
    if (NACC == 2) __syncthreads();
    if (threadIdx.x == 0) {
        sh.flags = 0u;
        dotEpilogue(mode, sh.sum[0], sh.sum[NACC - 1], &sh.ks, eps, tagOff, nullptr);
    }
    __syncthreads();
}

// the workgroup's maximum (>= 0) and change indicator, in every thread
__device__ __forceinline__ void smallJoin(SmallShared& sh, double& mx, bool& change)
{
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    mx = waveMax(mx);
    const bool any = __ballot(change) != 0ull;
    if (lane == 0) { sh.wmax[w] = mx; sh.wany[w] = any ? 1u : 0u; }
    __syncthreads();
    mx = 0.0;
    unsigned a = 0u;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) { mx = fmax(mx, sh.wmax[q]); a |= sh.wany[q]; }
    change = a != 0u;
}

template <int BS, class S>
__global__ __launch_bounds__(kThreads) void k_small_bicgstab(SmallArgs<S> a)
{
    __shared__ S sv[kSmallEntries];
    __shared__ SmallShared sh;
    const int m = BS * a.n, tid = (int)threadIdx.x;
    for (int k = tid; k < 2 * kAccLimbs; k += kThreads) sh.acc[k] = 0ull;
    if (tid == 0) sh.flags = 0u;
    // x = 0, r = b, p = v = 0, the initial norm
    double mx = 0.0;
    bool change = false;
#pragma unroll 1
    for (int i = tid; i < m; i += kThreads) {
        const S ri = a.b[i];
        a.x[i] = S(0); a.r[i] = ri; a.p[i] = S(0); a.v[i] = S(0);
        mx = fmax(mx, fabs((double)ri));
    }
    smallJoin(sh, mx, change);
    const double eps = (double)std::numeric_limits<S>::min() * 1e10;
    const double init = fmax(mx, eps);
    KrylovScalars& ks = sh.ks;
    if (tid == 0) {
        ks.rho = ks.alpha = ks.omega = 1.0;
        ks.beta = ks.rho_i = ks.denom = ks.resnorm = 0.0;
        ks.init_norm = init;
        ks.fail_code = 0; ks.fail_tag = -1; ks.stag_half = 0; ks.stag_full_tag = -1; ks.tag_base = 0; ks.iters = 0;
        ks.tol = a.tol; ks.abs_tol = a.absTol; ks.max_error = a.maxError;
        ks.run = 1; ks.stop_rc = -1; ks.stop_back = 0;
        if (init / fmax(1e-20, init) <= a.tol || init <= a.absTol) { ks.run = 0; ks.stop_rc = 0; }
    }
    __syncthreads();
    for (int it = 0; it < a.maxIter && ks.run; ++it) {
        // rho, p, y = M^-1 p, v = A y, alpha, the update and its test
        smallDot<S, 1>(m, a.b, a.r, sh, kDotRho, eps, 0);
        {
            const S omega = (S)ks.omega, beta = (S)ks.beta;
#pragma unroll 1
            for (int i = tid; i < m; i += kThreads) {
                S tmp = a.v[i];
                tmp *= omega;
                tmp -= a.p[i];
                tmp *= -beta;
                S pn = a.r[i];
                pn += tmp;
                a.p[i] = pn;
            }
        }
        __syncthreads();
        smallSweep<BS, S, false>(a, a.p, sv);
        smallSweep<BS, S, true>(a, nullptr, sv);
        smallSpmv<BS, S>(a, sv, a.v);
        smallDot<S, 1>(m, a.b, a.v, sh, kDotAlpha, eps, 0);
        {
            const S alpha = (S)ks.alpha;
            mx = 0.0;
            change = false;
#pragma unroll 1
            for (int i = tid; i < m; i += kThreads) {
                const S yi = sv[i];
                S tmp = yi;
                tmp *= alpha;
                tmp += a.x[i];
                a.x[i] = tmp;
                tmp = a.v[i];
                tmp *= alpha;
                S ri = a.r[i];
                ri -= tmp;
                a.r[i] = ri;
                mx = fmax(mx, fabs((double)ri));
                change |= yi != S(0);
            }
            smallJoin(sh, mx, change);
            if (tid == 0) {
                ks.iters = it;
                criterion(mx, change, &ks);
                if (!ks.run) ks.iters = it - ks.stop_back;
            }
            __syncthreads();
        }
        if (!ks.run) break;
        // z = M^-1 r, t = A z, omega, the update
        smallSweep<BS, S, false>(a, a.r, sv);
        smallSweep<BS, S, true>(a, nullptr, sv);
        smallSpmv<BS, S>(a, sv, a.t);
        smallDot<S, 2>(m, a.t, a.r, sh, kDotOmega, eps, 1);
        {
            const S omega = (S)ks.omega;
            change = false;
            mx = 0.0;
#pragma unroll 1
            for (int i = tid; i < m; i += kThreads) {
                const S zi = sv[i];
                a.x[i] += omega * zi;
                change |= zi != S(0);
                a.r[i] += -omega * a.t[i];
            }
            smallJoin(sh, mx, change);
            if (tid == 0) {
                if (!change && ks.stag_full_tag < 0) ks.stag_full_tag = ks.tag_base + 1;
                ks.tag_base += 2;
                ks.iters = it + 1;
            }
            __syncthreads();
        }
    }
    if (tid == 0) *a.ks = ks;
}

// ILU(0) by levels, BS lanes per row: lane e forms row e of the row's blocks
// (Dune's bilu0_decomposition in the operation order of k_ilu_factor_level).
// A level's time is a chain of loads from L2: for each lower neighbour its
// column, then that row's diagonal, end and inverted pivot, then the merge of
// the two rows, whose block the next neighbour or the pivot reads back.  With
// the one or two lower neighbours of the 48x32 lens problem 3.0 us a level (0.24 ms
// for 79 levels), against launches of 4.4 us each and the gaps between them.
template <int BS, class S>
__global__ __launch_bounds__(kThreads) void k_small_factor(int nLevels, int nChunks, const int4* __restrict__ slots,
    const int* __restrict__ rp, const int* __restrict__ ci, const int* __restrict__ diag, S* lu, double* __restrict__ dinv,
    int* __restrict__ fail)
{
    constexpr int LPR = RowLanes<BS>::kLanes, RPW = RowLanes<BS>::kRows, BB = BS * BS;
    const int lane = (int)(threadIdx.x & 63u), w = uniform((int)(threadIdx.x >> 6));
    const int e = lane % LPR, s = lane / LPR;
    const int4 none = make_int4(-1, 0, 0, -1);
    int t = w;
    slots += (long)RPW * LevelSchedule::kSlotPad + s;
    int4 m = t < nChunks ? slots[(long)t * RPW] : none;
    for (int l = 0; l < nLevels; ++l) {
        while (uniform(m.w) == l) {
            if (m.x >= 0 && e < BS) {
                const int i = m.x, kd = m.y + slotLower(m), k1 = kd + slotUpper(m) + 1;
                for (int ij = m.y; ij < kd; ++ij) {
                    const int j = ci[ij], jj = diag[j], je = rp[j + 1];
                    S Ar[BS], Lr[BS], Dj[BB];
#pragma unroll
                    for (int q = 0; q < BS; ++q) Ar[q] = lu[(long)BB * ij + BS * e + q];
#pragma unroll
                    for (int q = 0; q < BB; ++q) Dj[q] = lu[(long)BB * jj + q];
#pragma unroll
                    for (int c = 0; c < BS; ++c) {
                        S sum = Ar[0] * Dj[c];
#pragma unroll
                        for (int q = 1; q < BS; ++q) sum += Ar[q] * Dj[q * BS + c];
                        Lr[c] = sum;
                    }
#pragma unroll
                    for (int q = 0; q < BS; ++q) lu[(long)BB * ij + BS * e + q] = Lr[q];
                    int ik = ij + 1, jk = jj + 1;
                    while (ik < k1 && jk < je) {
                        const int cik = ci[ik], cjk = ci[jk];
                        if (cik == cjk) {
                            S Aj[BB];
#pragma unroll
                            for (int q = 0; q < BB; ++q) Aj[q] = lu[(long)BB * jk + q];
#pragma unroll
                            for (int c = 0; c < BS; ++c) {
                                S sum = Lr[0] * Aj[c];
#pragma unroll
                                for (int q = 1; q < BS; ++q) sum += Lr[q] * Aj[q * BS + c];
                                lu[(long)BB * ik + BS * e + c] -= sum;
                            }
                            ++ik; ++jk;
                        } else if (cik < cjk) ++ik;
                        else ++jk;
                    }
                }
                // the pivot: every lane of the row inverts the whole block and keeps its row
                S own[BS], P[BB];
#pragma unroll
                for (int q = 0; q < BS; ++q) own[q] = lu[(long)BB * kd + BS * e + q];
#pragma unroll
                for (int q = 0; q < BS; ++q) {
                    P[q] = rowComponent<BS, 0>(own[q]);
                    P[BS + q] = rowComponent<BS, 1>(own[q]);
                    if constexpr (BS == 3) P[2 * BS + q] = rowComponent<BS, 2>(own[q]);
                }
                if (!bInvert<BS, S>(P)) atomicOr(fail, 2);
#pragma unroll
                for (int r = 0; r < BS; ++r)
                    if (r == e) {
#pragma unroll
                        for (int q = 0; q < BS; ++q) {
                            lu[(long)BB * kd + BS * e + q] = P[r * BS + q];
                            dinv[(long)BB * i + BS * e + q] = (double)P[r * BS + q];
                        }
                    }
            }
            t += kWaves;
            m = t < nChunks ? slots[(long)t * RPW] : none;
        }
        __syncthreads();
    }
}

}  // namespace

template <class S>
void launchSmallBicgstab(int n, int bs, const LevelSchedule& L, const int* rp, const int* ci, const S* A, const S* lu,
                         const double* dinv, const S* b, S* x, S* const w[4], double tol, double absTol,
                         double maxError, int maxIter, KrylovScalars* ks, hipStream_t st)
{
    SmallArgs<S> a;
    a.n = n; a.nLevels = L.nLevels; a.nChunks = L.nChunks; a.maxIter = maxIter;
    a.slots = L.slots.p;
    a.rp = rp; a.ci = ci; a.A = A; a.lu = lu; a.dinv = dinv; a.b = b; a.x = x;
    a.r = w[0]; a.p = w[1]; a.v = w[2]; a.t = w[3];
    a.ks = ks;
    a.tol = tol; a.absTol = absTol; a.maxError = maxError;
    if (bs == 3) hipLaunchKernelGGL((k_small_bicgstab<3, S>), dim3(1), dim3(kThreads), 0, st, a);
    else hipLaunchKernelGGL((k_small_bicgstab<2, S>), dim3(1), dim3(kThreads), 0, st, a);
    OM_HIP(hipGetLastError());
}
template void launchSmallBicgstab<double>(int, int, const LevelSchedule&, const int*, const int*, const double*,
                                          const double*, const double*, const double*, double*, double* const[4],
                                          double, double, double, int, KrylovScalars*, hipStream_t);
template void launchSmallBicgstab<float>(int, int, const LevelSchedule&, const int*, const int*, const float*,
                                         const float*, const double*, const float*, float*, float* const[4], double,
                                         double, double, int, KrylovScalars*, hipStream_t);

template <class S>
void launchSmallFactor(int n, int bs, const LevelSchedule& L, const int* rp, const int* ci, const int* diag, S* lu,
                       double* dinv, int* dFail, hipStream_t st)
{
    (void)n;
    if (bs == 3)
        hipLaunchKernelGGL((k_small_factor<3, S>), dim3(1), dim3(kThreads), 0, st, L.nLevels, L.nChunks, L.slots.p, rp,
                           ci, diag, lu, dinv, dFail);
    else
        hipLaunchKernelGGL((k_small_factor<2, S>), dim3(1), dim3(kThreads), 0, st, L.nLevels, L.nChunks, L.slots.p, rp,
                           ci, diag, lu, dinv, dFail);
    OM_HIP(hipGetLastError());
}
template void launchSmallFactor<double>(int, int, const LevelSchedule&, const int*, const int*, const int*, double*,
                                        double*, int*, hipStream_t);
template void launchSmallFactor<float>(int, int, const LevelSchedule&, const int*, const int*, const int*, float*,
                                       double*, int*, hipStream_t);

}  // namespace omodels

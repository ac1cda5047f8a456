// exact_sum.h -- dot products whose result does not depend on the summation
// order: the products are added exactly into a long fixed-point accumulator
// and the sum is rounded once, to the nearest double (ties to even).
//
// The reference sums sequentially (OverlappingScalarProduct::dot,
// overlappingscalarproduct.hh:58-70, a plain loop over the entries); that
// result depends on the order of the additions, so a parallel reduction can
// only reproduce it by fixing the order.  The exact sum is the value the
// sequential loop approximates, it is the same for every partition of the
// work (one reservoir or a member of an ensemble, any grid size), and the CPU
// restatement computes the same value.
//
// Representation.  A finite double is m * 2^(pos - 1074) with an integer
// m < 2^53 and 0 <= pos <= 2045.  An accumulator holds kAccLimbs signed
// 64-bit limbs, limb j weighing 2^(32 j - 1074).  A product is cut at the
// limb boundary below it (k = pos / 32): the integer m * 2^(pos mod 32) <
// 2^85 goes as three chunks below 2^32 into limbs k, k+1, k+2.  Carries are
// deferred: with fewer than 2^28 products no limb can overflow.
//
// Reduction.  A wave splits each product error-free into four bands fixed
// by the wave's largest product (q = (sigma + r) - sigma, r -= q, for
// sigma = 2^(e_max + 10), 2^(e_max - 33), ...): every band's parts are
// multiples of its unit and their sum over the wave stays below 2^53 units,
// so the bands add exactly in double; a product with bits below the last
// band (2^-119 and less of the largest) adds its remainder to LDS directly.
// The wave's four band sums go into the workgroup's limbs in LDS (waves whose
// largest product is outside [2^-700, 2^1000] use a register window of
// integer limbs instead).  Each workgroup then adds its nonzero limbs to the
// device accumulator with device-scope atomics; the last workgroup to finish
// (a ticket counter) reads the accumulator, rounds, and clears it and the
// ticket for the next use.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace omodels {

constexpr int kAccLimbs = 68;      // 32-bit digits from 2^-1074; the largest product ends in digit 66

// The device accumulator of one sum: limbs with deferred carries and the
// non-finite products seen (1 NaN, 2 +inf, 4 -inf); zero between products.
struct ExactAcc {
    unsigned long long limb[kAccLimbs];
    unsigned int flags, pad_;
};

// One product placed in the accumulator: |p| = (hi * 2^64 + lo) * 2^(32 k - 1074)
// with hi * 2^64 + lo < 2^85; k < 0 for a zero or non-finite product.
struct ProductPiece {
    unsigned long long lo, hi;
    int k, neg;
};

__host__ __device__ __forceinline__ ProductPiece makePiece(double p, unsigned& flags)
{
    ProductPiece q;
    union { double d; unsigned long long u; } cv;
    cv.d = p;
    const unsigned long long b = cv.u;
    const int be = (int)((b >> 52) & 0x7ffu);
    unsigned long long man = b & 0xFFFFFFFFFFFFFull;
    q.neg = (int)(b >> 63);
    q.lo = 0ull; q.hi = 0ull; q.k = -1;
    if (be == 0x7ff) { flags |= man ? 1u : (q.neg ? 4u : 2u); return q; }
    if (be == 0 && man == 0ull) return q;
    int pos = 0;
    if (be) { man |= 1ull << 52; pos = be - 1; }
    q.k = pos >> 5;
    const int sh = pos & 31;
    q.lo = man << sh;
    q.hi = sh ? (man >> (64 - sh)) : 0ull;
    return q;
}

// The correctly rounded value of the accumulator.  d: the limbs as signed
// integers (overwritten), nonzero at most in [lo, hi]; flags as in ExactAcc.
__host__ __device__ inline double exactRound(long long* d, int lo, int hi, unsigned flags)
{
    union { double d; unsigned long long u; } cv;
    if ((flags & 1u) || (flags & 6u) == 6u) { cv.u = 0x7FF8000000000000ull; return cv.d; }
    if (flags & 2u) { cv.u = 0x7FF0000000000000ull; return cv.d; }
    if (flags & 4u) { cv.u = 0xFFF0000000000000ull; return cv.d; }
    if (lo > hi) return 0.0;
    // carries: digits in [0, 2^32), the sign in the carry out of digit hi + 1
    const int top = hi + 1 < kAccLimbs ? hi + 1 : kAccLimbs - 1;
    if (top > hi) d[top] = 0;
    long long carry = 0;
    for (int j = lo; j <= top; ++j) {
        const long long t = d[j] + carry;
        d[j] = t & 0xffffffffll;
        carry = t >> 32;
    }
    const bool neg = carry < 0;
    if (neg) {   // magnitude: two's complement of the digits
        long long c = 1;
        for (int j = lo; j <= top; ++j) {
            const long long t = (~d[j] & 0xffffffffll) + c;
            d[j] = t & 0xffffffffll;
            c = t >> 32;
        }
    }
    int h = top;
    while (h >= lo && d[h] == 0) --h;
    if (h < lo) return 0.0;
    const unsigned long long sgn = neg ? (1ull << 63) : 0ull;
    int lz = 0;
    for (unsigned long long v = (unsigned long long)d[h]; !(v & 0x80000000ull); v <<= 1) ++lz;
    int b = 32 * h + 31 - lz;       // leading bit, in units of 2^-1074
    if (b < 53) {                   // subnormal or smallest normal: exact
        unsigned long long v = 0ull;
        for (int j = h; j >= lo; --j) v = (v << 32) | (unsigned long long)d[j];
        v <<= 32 * lo;
        cv.u = sgn | v;
        return cv.d;
    }
    // the 64 bits ending at the leading bit, and whether anything lies below them
    auto dig = [&](int j) -> unsigned long long { return (j >= lo && j <= top) ? (unsigned long long)d[j] : 0ull; };
    const int s = 32 - lz;          // bits of digit h - 2 below the window
    const unsigned long long hiw = dig(h), midw = dig(h - 1), low = dig(h - 2);
    // window = (hiw * 2^64 + midw * 2^32 + low) >> s, s in [1, 32]
    const unsigned long long w = (hiw << (64 - s)) | (midw << (32 - s)) | (low >> s);
    bool sticky = (low & ((1ull << s) - 1ull)) != 0ull;
    for (int j = h - 3; j >= lo && !sticky; --j) sticky = d[j] != 0;
    unsigned long long mant = w >> 11;
    const bool rbit = (w >> 10) & 1ull;
    const bool rest = (w & 0x3ffull) != 0ull || sticky;
    if (rbit && (rest || (mant & 1ull))) ++mant;
    if (mant >> 53) { mant >>= 1; ++b; }
    const int biased = b - 51;
    if (biased >= 2047) { cv.u = sgn | 0x7FF0000000000000ull; return cv.d; }
    cv.u = sgn | ((unsigned long long)biased << 52) | (mant & 0xFFFFFFFFFFFFFull);
    return cv.d;
}

#ifdef __HIPCC__
// Reductions over a wave by DPP moves (row shifts, then the two row
// broadcasts): the result is lane 63's.  Absent lanes contribute zero bits.
template <int Ctrl, int RowMask>
__device__ __forceinline__ unsigned dppMove(unsigned x)
{
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, Ctrl, RowMask, 0xf, false);
}
template <int Ctrl, int RowMask>
__device__ __forceinline__ double dppMove(double x)
{
    return __hiloint2double((int)dppMove<Ctrl, RowMask>((unsigned)__double2hiint(x)),
                            (int)dppMove<Ctrl, RowMask>((unsigned)__double2loint(x)));
}
// the wave's sum in every lane; for sums that are exact in every order
__device__ __forceinline__ double waveSumExact(double v)
{
    v += dppMove<0x111, 0xf>(v);     // row_shr:1, 2, 4, 8
    v += dppMove<0x112, 0xf>(v);
    v += dppMove<0x114, 0xf>(v);
    v += dppMove<0x118, 0xf>(v);
    v += dppMove<0x142, 0xa>(v);     // row_bcast:15 into rows 1 and 3
    v += dppMove<0x143, 0xc>(v);     // row_bcast:31 into rows 2 and 3
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}
__device__ __forceinline__ unsigned waveMaxU(unsigned v)
{
    v = max(v, dppMove<0x111, 0xf>(v));
    v = max(v, dppMove<0x112, 0xf>(v));
    v = max(v, dppMove<0x114, 0xf>(v));
    v = max(v, dppMove<0x118, 0xf>(v));
    v = max(v, dppMove<0x142, 0xa>(v));
    v = max(v, dppMove<0x143, 0xc>(v));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

constexpr int kWindow = 8;      // limbs of a wave's register window (256 bits)

// Adds U products per lane of a wave to the workgroup's limbs sAcc (LDS,
// kAccLimbs).  Every lane of the wave must call it (absent products: 0.0).
template <int U>
__device__ __forceinline__ void accumulateWave(const double (&p)[U], unsigned long long* sAcc, unsigned& flags)
{
    int k[U];
    unsigned long long c0[U], c1[U], c2[U];
    int kmax = -1;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const ProductPiece q = makePiece(p[u], flags);
        k[u] = q.k;
        c0[u] = q.lo & 0xffffffffull; c1[u] = q.lo >> 32; c2[u] = q.hi;
        if (q.neg) { c0[u] = 0ull - c0[u]; c1[u] = 0ull - c1[u]; c2[u] = 0ull - c2[u]; }
        kmax = max(kmax, q.k);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) kmax = max(kmax, __shfl_xor(kmax, o, 64));
    if (kmax < 0) return;                        // wave-uniform: no nonzero finite product
    const int kb = kmax + 3 - kWindow;           // absolute limb of window limb 0
    unsigned long long acc[kWindow];
#pragma unroll
    for (int w = 0; w < kWindow; ++w) acc[w] = 0ull;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (k[u] < 0) continue;
        const int t = k[u] - kb;
        if (t >= 0) {
#pragma unroll
            for (int w = 0; w < kWindow; ++w)
                acc[w] += w == t ? c0[u] : (w == t + 1 ? c1[u] : (w == t + 2 ? c2[u] : 0ull));
        } else {                                 // far below the wave's largest product
            atomicAdd(&sAcc[k[u]], c0[u]);
            atomicAdd(&sAcc[k[u] + 1], c1[u]);
            atomicAdd(&sAcc[k[u] + 2], c2[u]);
        }
    }
#pragma unroll
    for (int w = 0; w < kWindow; ++w)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc[w] += __shfl_xor(acc[w], o, 64);
    const int lane = (int)(threadIdx.x & 63u);
    unsigned long long v = 0ull;
#pragma unroll
    for (int w = 0; w < kWindow; ++w) v = lane == w ? acc[w] : v;
    if (lane < kWindow && v && kb + lane >= 0) atomicAdd(&sAcc[kb + lane], v);
}

// one value's chunks straight into LDS limbs
__device__ __forceinline__ void addToLimbs(double v, unsigned long long* sAcc, unsigned& flags)
{
    const ProductPiece q = makePiece(v, flags);
    if (q.k < 0) return;
    unsigned long long c0 = q.lo & 0xffffffffull, c1 = q.lo >> 32, c2 = q.hi;
    if (q.neg) { c0 = 0ull - c0; c1 = 0ull - c1; c2 = 0ull - c2; }
    atomicAdd(&sAcc[q.k], c0);
    atomicAdd(&sAcc[q.k + 1], c1);
    if (c2) atomicAdd(&sAcc[q.k + 2], c2);
}

// Adds U products per lane of a wave to the workgroup's limbs sAcc (LDS) by
// the error-free band split.  Every lane of the wave must call it (absent
// products: 0.0); U <= 64.
template <int U>
__device__ __forceinline__ void accumulateBands(const double (&p)[U], unsigned long long* sAcc, unsigned& flags)
{
    unsigned be = 0u;            // the largest biased exponent of a finite product
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const unsigned e = ((unsigned)__double2hiint(p[u]) >> 20) & 0x7ffu;
        be = max(be, e == 0x7ffu ? 0u : e);
    }
    be = waveMaxU(be);
    if (be < 1023u - 700u || be > 1023u + 1000u) {     // no finite nonzero product, or extreme ones
        accumulateWave<U>(p, sAcc, flags);
        return;
    }
    constexpr int kBands = 4;
    double S[kBands];
#pragma unroll
    for (int i = 0; i < kBands; ++i) S[i] = 0.0;
    const double sigma0 = __hiloint2double((int)((be + 10u) << 20), 0);     // 2^(e_max + 10)
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (!isfinite(p[u])) { addToLimbs(p[u], sAcc, flags); continue; }
        double r = p[u], sigma = sigma0;
#pragma unroll
        for (int i = 0; i < kBands; ++i) {
            const double q = (sigma + r) - sigma;
            S[i] += q;
            r -= q;
            sigma *= 0x1p-43;
        }
        if (r != 0.0) addToLimbs(r, sAcc, flags);
    }
#pragma unroll
    for (int i = 0; i < kBands; ++i) S[i] = waveSumExact(S[i]);
    const int lane = (int)(threadIdx.x & 63u);
    if (lane < kBands) {
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < kBands; ++i) v = lane == i ? S[i] : v;
        addToLimbs(v, sAcc, flags);
    }
}

// The workgroup's limbs of nAcc sums (LDS, nAcc * kAccLimbs) and their flags
// (3 bits each) in sMeta[0]; sMeta[1] belongs to lastToFinish.
__device__ __forceinline__ void clearLimbs(unsigned long long* sAcc, int nAcc, unsigned* sMeta)
{
    for (int t = (int)threadIdx.x; t < nAcc * kAccLimbs; t += (int)blockDim.x) sAcc[t] = 0ull;
    if (threadIdx.x == 0) sMeta[0] = 0u;
}

// Adds the workgroup's limbs of nAcc sums to the device accumulators g[0..nAcc)
// (after the barrier that ends the accumulation).
__device__ __forceinline__ void flushLimbs(const unsigned long long* sAcc, int nAcc, const unsigned* sMeta,
                                           ExactAcc* g)
{
    for (int t = (int)threadIdx.x; t < nAcc * kAccLimbs; t += (int)blockDim.x) {
        const unsigned long long v = sAcc[t];
        if (v) __hip_atomic_fetch_add(&g[t / kAccLimbs].limb[t % kAccLimbs], v, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
    }
    if (threadIdx.x == 0 && sMeta[0])
        for (int a = 0; a < nAcc; ++a) {
            const unsigned f = (sMeta[0] >> (3 * a)) & 7u;
            if (f) __hip_atomic_fetch_or(&g[a].flags, f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
}

// After every thread's atomics: true in every thread of the workgroup that
// finishes last among nBlocks; that workgroup resets the ticket.
__device__ __forceinline__ bool lastToFinish(unsigned* ticket, int nBlocks, unsigned* sMeta)
{
    __builtin_amdgcn_s_waitcnt(0x0F70);     // this wave's atomics acknowledged
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = t == (unsigned)nBlocks - 1u;
        if (last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sMeta[1] = last ? 1u : 0u;
    }
    __syncthreads();
    return sMeta[1] != 0u;
}

// For one thread of each workgroup of a grid, its result acknowledged: true in
// the last one.  Many workgroups meet in kFinishGroups groups first, whose
// tickets lie in lines of their own.  Atomics on one word pass at about 13 ns
// each, so 256 workgroups on one ticket take 3.3 us; the groups' second round
// trip takes 1 us, which fewer than 64 workgroups would not win back.  The
// last one resets the tickets.
constexpr int kFinishGroups = 16, kFinishFlat = 64;
struct alignas(128) FinishTicket {
    unsigned n;
};
__device__ __forceinline__ bool takeTicket(FinishTicket* t, int count)
{
    if (__hip_atomic_fetch_add(&t->n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != (unsigned)count - 1u) return false;
    __hip_atomic_store(&t->n, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}
// tickets: kFinishGroups + 1, the last one the groups' own
__device__ __forceinline__ bool lastTicketOfGrid(FinishTicket* tickets)
{
    const int nb = (int)gridDim.x, G = nb > kFinishFlat ? kFinishGroups : 1, g = (int)blockIdx.x % G;
    return takeTicket(&tickets[g], (nb - g + G - 1) / G) && (G == 1 || takeTicket(&tickets[kFinishGroups], G));
}

// exactRound by one wave: lane j holds limb j as a signed integer, and limbs
// 62 and up are zero.  Every lane gets the value.
__device__ __forceinline__ double waveRound(long long limb, unsigned flags)
{
    if ((flags & 1u) || (flags & 6u) == 6u) return __longlong_as_double(0x7FF8000000000000ll);
    if (flags & 2u) return __longlong_as_double(0x7FF0000000000000ll);
    if (flags & 4u) return __longlong_as_double((long long)0xFFF0000000000000ull);
    const unsigned long long nz = __ballot(limb != 0);
    if (!nz) return 0.0;
    const int lane = (int)(threadIdx.x & 63u);
    const int lo = __builtin_ctzll(nz), top = 64 - __builtin_clzll(nz);      // one above the last nonzero limb
    unsigned dg = 0u;               // lane j: digit j of the magnitude
    bool neg = false;
    for (int pass = 0; pass < 2; ++pass) {
        long long carry = 0;
        for (int j = lo; j <= top; ++j) {
            const unsigned wl = (unsigned)__builtin_amdgcn_readlane((int)limb, j);
            const int wh = __builtin_amdgcn_readlane((int)(limb >> 32), j);
            const long long t = (long long)(((unsigned long long)(unsigned)wh << 32) | wl) + carry;
            dg = lane == j ? (unsigned)t : dg;
            carry = t >> 32;
        }
        if (carry >= 0) break;
        neg = true;                 // the magnitude: the digits of the negated limbs
        limb = -limb;
    }
    const unsigned long long dz = __ballot(dg != 0u);
    if (!dz) return 0.0;
    const int h = 63 - __builtin_clzll(dz);
    auto dig = [&](int j) -> unsigned long long {
        return j < 0 ? 0ull : (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)dg, j);
    };
    const unsigned long long sgn = neg ? (1ull << 63) : 0ull;
    const unsigned long long hiw = dig(h), midw = dig(h - 1), low = dig(h - 2);
    const int lz = __builtin_clz((unsigned)hiw);
    int b = 32 * h + 31 - lz;       // leading bit, in units of 2^-1074
    if (b < 53)                     // subnormal or smallest normal: exact
        return __longlong_as_double((long long)(sgn | (dig(1) << 32) | dig(0)));
    const int s = 32 - lz;          // bits of digit h - 2 below the window of 64
    const unsigned long long w = (hiw << (64 - s)) | (midw << (32 - s)) | (low >> s);
    const bool below = h > 2 && (dz & ((1ull << (h - 2)) - 1ull)) != 0ull;
    const bool sticky = (low & ((1ull << s) - 1ull)) != 0ull || below;
    unsigned long long mant = w >> 11;
    if (((w >> 10) & 1ull) && ((w & 0x3ffull) != 0ull || sticky || (mant & 1ull))) ++mant;
    if (mant >> 53) { mant >>= 1; ++b; }
    const int biased = b - 51;
    if (biased >= 2047) return __longlong_as_double((long long)(sgn | 0x7FF0000000000000ull));
    return __longlong_as_double((long long)(sgn | ((unsigned long long)biased << 52) | (mant & 0xFFFFFFFFFFFFFull)));
}

// The rounded value of an accumulator in one wave's registers: v0 limb
// `lane`, v1 limb 64 + lane (zero where there is none).
__device__ __forceinline__ double roundLimbs(unsigned long long v0, unsigned long long v1, unsigned flags,
                                             long long* sD)
{
    const int lane = (int)(threadIdx.x & 63u);
    if (__ballot(v1 != 0ull || (lane >= 62 && v0 != 0ull)) == 0ull) return waveRound((long long)v0, flags);
    // products of 2^910 and more: one thread over LDS
    sD[lane] = (long long)v0;
    if (lane + 64 < kAccLimbs) sD[lane + 64] = (long long)v1;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    double r = 0.0;
    if (lane == 0) {
        int lo = kAccLimbs, hi = -1;
        for (int t = 0; t < kAccLimbs; ++t)
            if (sD[t]) { if (lo == kAccLimbs) lo = t; hi = t; }
        r = exactRound(sD, lo, hi, flags);
    }
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(r)),
                            __builtin_amdgcn_readfirstlane(__double2loint(r)));
}

// In one wave of the last workgroup: the rounded value of the device
// accumulator g, which is cleared for the next use; every lane gets it.  sD:
// LDS of kAccLimbs long longs of this wave's own.  The chain of carries over
// the limbs bounds it: it runs through readlane and scalar adds instead of one
// thread's LDS accesses, 0.6 us instead of 3.0 us per sum.
__device__ __forceinline__ double finishExact(ExactAcc* g, long long* sD)
{
    const int lane = (int)(threadIdx.x & 63u);
    const bool two = lane + 64 < kAccLimbs;
    const unsigned long long v0 = __hip_atomic_load(&g->limb[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long v1 =
        two ? __hip_atomic_load(&g->limb[lane + 64], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
    const unsigned flags = (unsigned)__builtin_amdgcn_readfirstlane(
        (int)__hip_atomic_load(&g->flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (v0) __hip_atomic_store(&g->limb[lane], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v1) __hip_atomic_store(&g->limb[lane + 64], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (flags && lane == 0) __hip_atomic_store(&g->flags, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return roundLimbs(v0, v1, flags, sD);
}

// In the last workgroup (at least NACC waves): the sums g[0..NACC) in every
// thread of wave 0; one wave per sum.
template <int NACC>
__device__ __forceinline__ void finishSums(ExactAcc* g, double (&sum)[2])
{
    __shared__ long long sD[NACC * kAccLimbs];
    __shared__ double sR[NACC];
    const int w = (int)(threadIdx.x >> 6);
    sum[0] = sum[1] = 0.0;
    if (w < NACC) {
        sum[0] = finishExact(g + w, sD + w * kAccLimbs);
        sR[w] = sum[0];
    }
    if (NACC == 1) return;
    __syncthreads();
    sum[0] = sR[0];
    sum[1] = sR[NACC - 1];
}
#endif

}  // namespace omodels

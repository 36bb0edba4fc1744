// qk_kernels.h -- device code shared by the per-class translation units.
#pragma once
#include <utility>
#include "qk_internal.h"
#include "eri_generated.inc"

namespace qk {

__host__ __device__ constexpr int ncart(int l) { return (l + 1) * (l + 2) / 2; }
__host__ __device__ constexpr int nrange(int lo, int hi) {
    return hi < lo ? 0 : ncart(hi) + nrange(lo, hi - 1);
}

// QUICK's FmT (subs/fmt.f90:12-84; gpu_get2e_subs.h:1386-1457) restated: the
// piecewise fit of F_0 (or F_Mb near T = 0), then upward recursion for
// T > 3e-5 (T > 3e-7 when Mb < 4), else downward recursion from Mb.  Mb is the
// order the reference asks for; values F_0..F_LT are produced (LT <= Mb).
template <int LT>
__device__ __forceinline__ void boys_ref(double X, int Mb, double* F) {
    const double PIE4 = 3.1415926535897932384626433832795 / 4.0;
    const double E = exp(-X);
    const bool up = (X > 3.0e-5) || (X > 3.0e-7 && Mb < 4);
    if (up) {
        const double XINV = 1.0 / X;
        double WW1;
        if (X > 5.0) {
            const double s = sqrt(PIE4 * XINV);
            if (X > 33.0) {
                WW1 = s;
            } else if (X > 15.0) {
                WW1 = ((1.9623264149430e-01 * XINV - 4.9695241464490e-01) * XINV - 6.0156581186481e-05) * E + s;
            } else if (X > 10.0) {
                WW1 = (((-1.8784686463512e-01 * XINV + 2.2991849164985e-01) * XINV - 4.9893752514047e-01) * XINV -
                       2.1916512131607e-05) * E + s;
            } else {
                WW1 = ((((((4.6897511375022e-01 * XINV - 6.9955602298985e-01) * XINV + 5.3689283271887e-01) * XINV -
                          3.2883030418398e-01) * XINV + 2.4645596956002e-01) * XINV - 4.9984072848436e-01) * XINV -
                       3.1501078774085e-06) * E + s;
            }
        } else if (X > 1.0) {
            double F1;
            if (X > 3.0) {
                const double Y = X - 4.0;
                F1 = ((((((((((-2.62453564772299e-11 * Y + 3.24031041623823e-10) * Y - 3.614965656163e-09) * Y +
                             3.760256799971e-08) * Y - 3.553558319675e-07) * Y + 3.022556449731e-06) * Y -
                          2.290098979647e-05) * Y + 1.526537461148e-04) * Y - 8.81947375894379e-04) * Y +
                       4.33207949514611e-03) * Y - 1.75257821619926e-02) * Y + 5.28406320615584e-02;
            } else {
                const double Y = X - 2.0;
                F1 = ((((((((((-1.61702782425558e-10 * Y + 1.96215250865776e-09) * Y - 2.14234468198419e-08) * Y +
                             2.17216556336318e-07) * Y - 1.98850171329371e-06) * Y + 1.62429321438911e-05) * Y -
                          1.16740298039895e-04) * Y + 7.24888732052332e-04) * Y - 3.79490003707156e-03) * Y +
                       1.61723488664661e-02) * Y - 5.29428148329736e-02) * Y + 1.15702180856167e-01;
            }
            WW1 = (X + X) * F1 + E;
        } else {
            const double F1 = ((((((((-8.36313918003957e-08 * X + 1.21222603512827e-06) * X - 1.15662609053481e-05) * X +
                                    9.25197374512647e-05) * X - 6.40994113129432e-04) * X + 3.78787044215009e-03) * X -
                                 1.85185172458485e-02) * X + 7.14285713298222e-02) * X - 1.99999999997023e-01) * X +
                              3.33333333333318e-01;
            WW1 = (X + X) * F1 + E;
        }
        F[0] = WW1;
#pragma unroll
        for (int m = 1; m <= LT; ++m) F[m] = (double(2 * m - 1) * F[m - 1] - E) * 0.5 * XINV;
    } else {
        double v = (1.0 - X) / double(2 * Mb + 1);
        const double twot = X * 2.0;
        for (int m = Mb - 1; m >= LT; --m) v = (twot * v + E) / double(m * 2 + 1);
        F[LT] = v;
#pragma unroll
        for (int m = LT - 1; m >= 0; --m) F[m] = (twot * F[m + 1] + E) / double(m * 2 + 1);
    }
}

// The same fit without branches on T: the seven regions' polynomials, zero-padded
// to 12 coefficients (highest power first), are evaluated by one Horner chain
// over coefficients read from a per-block copy of kBoysFit; the padding makes
// every region's chain identical to its own shorter one (fma(0, z, c) = c), and
// F_0 = fma(v, u, w) with (z, u, w) = (X, 2X, E), (X-2, 2X, E), (X-4, 2X, E) below
// T = 5 and (1/X, E, sqrt(pi/4X)) above.  Lanes of a wavefront with different T
// then execute one path instead of one per region.
constexpr int kBoysFitRegions = 7, kBoysFitTerms = 12;
__constant__ const double kBoysFit[kBoysFitRegions * kBoysFitTerms] = {
    0, 0, -8.36313918003957e-08, 1.21222603512827e-06, -1.15662609053481e-05, 9.25197374512647e-05,
    -6.40994113129432e-04, 3.78787044215009e-03, -1.85185172458485e-02, 7.14285713298222e-02,
    -1.99999999997023e-01, 3.33333333333318e-01,
    -1.61702782425558e-10, 1.96215250865776e-09, -2.14234468198419e-08, 2.17216556336318e-07,
    -1.98850171329371e-06, 1.62429321438911e-05, -1.16740298039895e-04, 7.24888732052332e-04,
    -3.79490003707156e-03, 1.61723488664661e-02, -5.29428148329736e-02, 1.15702180856167e-01,
    -2.62453564772299e-11, 3.24031041623823e-10, -3.614965656163e-09, 3.760256799971e-08,
    -3.553558319675e-07, 3.022556449731e-06, -2.290098979647e-05, 1.526537461148e-04,
    -8.81947375894379e-04, 4.33207949514611e-03, -1.75257821619926e-02, 5.28406320615584e-02,
    0, 0, 0, 0, 0, 4.6897511375022e-01, -6.9955602298985e-01, 5.3689283271887e-01, -3.2883030418398e-01,
    2.4645596956002e-01, -4.9984072848436e-01, -3.1501078774085e-06,
    0, 0, 0, 0, 0, 0, 0, 0, -1.8784686463512e-01, 2.2991849164985e-01, -4.9893752514047e-01, -2.1916512131607e-05,
    0, 0, 0, 0, 0, 0, 0, 0, 0, 1.9623264149430e-01, -4.9695241464490e-01, -6.0156581186481e-05,
    0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

// 1/sqrt(x) for the positive exponent sums of a primitive quartet: the hardware
// estimate refined by two Newton steps, y <- y + y (1 - x y^2) / 2, each of which
// squares the relative error (FP64); the hardware estimate (FP32, whose error
// budget is 1e-6).  A primitive quartet takes 1/(zeta+eta) as its square (one
// rounding more).
__device__ __forceinline__ double rsqrt_nr(double x) {
    double y = __builtin_amdgcn_rsq(x);
    y = fma(y * 0.5, fma(-x * y, y, 1.0), y);
    return fma(y * 0.5, fma(-x * y, y, 1.0), y);
}
__device__ __forceinline__ float rsqrt_nr(float x) { return __builtin_amdgcn_rsqf(x); }

// exp(-X), X >= 0: X = -k ln2 - r with |r| <= ln2 / 2 (ln2 in the two parts of
// fdlibm's e_exp.c, by Sun Microsystems: the high one exact times k below 2^21), exp(r) by the degree-11 interpolant at the
// Chebyshev nodes of the interval (largest relative error 1.7e-17), scaled by 2^k
// (to zero beyond the range; X up to 1e44, where r's error would overflow p)
__device__ __forceinline__ double exp_neg(double X) {
    const double k = __builtin_rint(X * -1.4426950408889634);
    const double r = fma(k, -1.9082149292705877e-10, fma(k, -0.6931471803691238, -X));
    double p = 2.511003761756205e-08;
    p = fma(p, r, 2.7632639654123758e-07);
    p = fma(p, r, 2.7557240918547625e-06);
    p = fma(p, r, 2.4801485482287731e-05);
    p = fma(p, r, 0.00019841269890047143);
    p = fma(p, r, 0.0013888888952314812);
    p = fma(p, r, 0.0083333333333196011);
    p = fma(p, r, 0.041666666666488092);
    p = fma(p, r, 0.1666666666666668);
    p = fma(p, r, 0.50000000000000189);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return __builtin_amdgcn_ldexp(p, int(k));
}

// QUICK's fit in two parts: the regions above T = 3e-5 (or 3e-7) without any
// branch, so that several primitive quartets can be interleaved, and the few
// lanes near T = 0 (centres that coincide) afterwards.
template <int LT>
__device__ __forceinline__ void boys_fit_main(double X, double E, const double* __restrict__ tab, double* F) {
    const double RS = rsqrt_nr(X);           // 1/sqrt(X); 1/X as its square
    const double XINV = RS * RS;
    const int r = int(X > 1.0) + int(X > 3.0) + int(X > 5.0) + int(X > 10.0) + int(X > 15.0) + int(X > 33.0);
    const double off = r == 0 ? 0.0 : (r == 1 ? 2.0 : 4.0);
    const double z = r <= 2 ? X - off : XINV;
    const double* c = tab + kBoysFitTerms * r;
    double v = c[0];
#pragma unroll
    for (int k = 1; k < kBoysFitTerms; ++k) v = fma(v, z, c[k]);
    const double s = 0.88622692545275801365 * RS;   // sqrt(PIE4 / X), sqrt(pi/4) = 0.886...
    F[0] = r <= 2 ? fma(v, X + X, E) : fma(v, E, s);
    const double h = 0.5 * XINV;
#pragma unroll
    for (int m = 1; m <= LT; ++m) F[m] = (double(2 * m - 1) * F[m - 1] - E) * h;
}
__device__ __forceinline__ bool boys_fit_up(double X, int Mb) { return (X > 3.0e-5) || (X > 3.0e-7 && Mb < 4); }
template <int LT>
__device__ __forceinline__ void boys_fit_near0(double X, double E, int Mb, double* F) {
    double v = (1.0 - X) / double(2 * Mb + 1);
    const double twot = X * 2.0;
    for (int m = Mb - 1; m >= LT; --m) v = (twot * v + E) / double(m * 2 + 1);
    F[LT] = v;
#pragma unroll
    for (int m = LT - 1; m >= 0; --m) F[m] = (twot * F[m + 1] + E) / double(m * 2 + 1);
}
template <int LT>
__device__ __forceinline__ void boys_fit(double X, int Mb, const double* __restrict__ tab, double* F) {
    const double E = exp_neg(X);
    boys_fit_main<LT>(X, E, tab, F);
    if (!boys_fit_up(X, Mb)) boys_fit_near0<LT>(X, E, Mb, F);
}

// Copies primitive pairs base, base + stride, ... (n <= 64 of them) into the
// wavefront's slab: field f of pair i at slab[f * 64 + i] (zeta, 1/2zeta, P, K,
// cutprim).  Every lane of the wavefront takes part; the fences order the slab's
// earlier reads before these writes and these writes before later reads (LDS
// operations of one wavefront complete in order).
template <class PP, typename R>
__device__ __forceinline__ void stage_bra(const PP& pp, int base, int stride, int n, int lane, R* slab) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < n) {
        const int k = base + lane * stride;
        slab[lane] = pp.zeta[k];
        slab[64 + lane] = pp.oo2z[k];
        slab[2 * 64 + lane] = pp.Px[k];
        slab[3 * 64 + lane] = pp.Py[k];
        slab[4 * 64 + lane] = pp.Pz[k];
        slab[5 * 64 + lane] = pp.K[k];
        slab[6 * 64 + lane] = pp.cut[k];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void fx_add(unsigned long long* X, long long idx, double v) {
    const long long iv = __double2ll_rn(v * 0x1p48);
    if (iv != 0) atomicAdd(X + idx, (unsigned long long)iv);
}

// round(v * 2^48) for |v| < 2^15 in FP32 arithmetic: with a = v 2^16 (exact),
// its integer part h = trunc(a) and fraction f = a - h (exact: the low bits of
// a, |f| <= 1 - 2^-24), the result is h 2^32 + rint(f 2^32); as h 2^32 is even
// and rint is odd-symmetric, this is the integer __double2ll_rn(double(v) *
// 0x1p48) gives, without FP64 instructions
__device__ __forceinline__ long long fx_round_f(float v) {
    const float a = v * 65536.0f;
    const float h = truncf(a);
    const unsigned lo = (unsigned)rintf(fabsf(a - h) * 4294967296.0f);
    const long long hi = (long long)(int)h * 4294967296LL;
    return a < 0.0f ? hi - (long long)lo : hi + (long long)lo;
}

__device__ __forceinline__ double dn_max(const double* cm, int ns, int A, int B, int C, int D) {
    double m = fmax(4.0 * cm[A * ns + B], 4.0 * cm[C * ns + D]);
    m = fmax(m, fmax(fmax(cm[A * ns + D], cm[A * ns + C]), fmax(cm[B * ns + C], cm[B * ns + D])));
    return m;
}

template <int LA, int LB, int LC, int LD>
struct ClassOps;

#define QK_CLASS(la, lb, lc, ld, TAG)                                                                    \
    template <>                                                                                          \
    struct ClassOps<la, lb, lc, ld> {                                                                    \
        template <typename R>                                                                            \
        static __device__ __forceinline__ void vrr(const R* F, R PAx, R PAy, R PAz, R WPx, R WPy, R WPz, \
                                                   R QCx, R QCy, R QCz, R WQx, R WQy, R WQz, R oo2z,     \
                                                   R oo2e, R oo2ze, R roz, R roe, R* acc) {              \
            vrr_##TAG<R>(F, PAx, PAy, PAz, WPx, WPy, WPz, QCx, QCy, QCz, WQx, WQy, WQz, oo2z, oo2e,      \
                         oo2ze, roz, roe, acc);                                                          \
        }                                                                                                \
        template <typename R>                                                                            \
        static __device__ __forceinline__ void hrr(const R* acc, R ABx, R ABy, R ABz, R CDx, R CDy,      \
                                                   R CDz, R* out) {                                      \
            hrr_##TAG<R>(acc, ABx, ABy, ABz, CDx, CDy, CDz, out);                                        \
        }                                                                                                \
    };

QK_CLASS(0, 0, 0, 0, ssss)
QK_CLASS(1, 0, 0, 0, psss)
QK_CLASS(1, 0, 1, 0, psps)
QK_CLASS(1, 1, 0, 0, ppss)
QK_CLASS(1, 1, 1, 0, ppps)
QK_CLASS(1, 1, 1, 1, pppp)
QK_CLASS(2, 0, 0, 0, dsss)
QK_CLASS(2, 0, 1, 0, dsps)
QK_CLASS(2, 0, 1, 1, dspp)
QK_CLASS(2, 0, 2, 0, dsds)
QK_CLASS(2, 1, 0, 0, dpss)
QK_CLASS(2, 1, 1, 0, dpps)
QK_CLASS(2, 1, 1, 1, dppp)
QK_CLASS(2, 1, 2, 0, dpds)
QK_CLASS(2, 1, 2, 1, dpdp)
QK_CLASS(2, 2, 0, 0, ddss)
QK_CLASS(2, 2, 1, 0, ddps)
QK_CLASS(2, 2, 1, 1, ddpp)
QK_CLASS(2, 2, 2, 0, ddds)
QK_CLASS(2, 2, 2, 1, dddp)
QK_CLASS(2, 2, 2, 2, dddd)

// Wavefronts per SIMD the light kernels are compiled for: two (256 VGPRs, no
// spills for the small accumulators), one for the larger classes.
template <int LA, int LB, int LC, int LD>
struct Occupancy {
    static constexpr int nacc = nrange(LA, LA + LB) * nrange(LC, LC + LD);
    static constexpr int value = nacc <= 36 ? 2 : 1;
};

// int64 sum over the 64 lanes of a wavefront (exact, so order-free)
__device__ __forceinline__ long long wave_sum_i64(long long v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// ---------------------------------------------------------------------------
// The thread-per-quartet Fock kernels: one body, in FP64 (fock_kernel) and in
// FP32 with FP64-grade accumulation (fock_kernel_f32).

// f(0), ..., f(N - 1) with compile-time arguments
template <class F, int... I>
__device__ __forceinline__ void for_each_int(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}

// pieces that differ with the arithmetic type
template <typename R>
struct FockType;
template <>
struct FockType<double> {
    static __device__ __forceinline__ const DevPrims& prims(const FockArgs& a) { return a.pp; }
    static __device__ __forceinline__ const double* density(const FockArgs& a) { return a.Dp; }
    static __device__ __forceinline__ long long fixed(double v) { return __double2ll_rn(v * 0x1p48); }
};
template <>
struct FockType<float> {
    static __device__ __forceinline__ const DevPrimsF& prims(const FockArgs& a) { return a.ppf; }
    static __device__ __forceinline__ const float* density(const FockArgs& a) { return a.Dpf; }
    static __device__ __forceinline__ long long fixed(float v) { return fx_round_f(v); }
};

// What a lane needs of a ket beyond its pair record, gathered ahead: the five
// shell-block density maxima of its screen, the centre C, its first primitive
template <typename R>
struct KetGather {
    double cd, ad, ac, bd, bc;
    double Cx, Cy, Cz;
    R z, o, x, y, zz, K, c;
};

// A wavefront takes tiles (a bra pair, up to 64 kets of one group, one per
// lane) t0, t0 + step, ... < t1.  Two thirds of its cycles used to go to waiting
// for memory: a tile's ket list, the kets' pair arrays, their Qshells' arrays,
// the density maxima and centres, and the primitives were five dependent
// round trips.  A pair's data now sits in one 32-byte record, and the next
// tiles are fetched while one is evaluated: the tile after next, the next tile's
// kets, and their records at the top; their screens, centres and first
// primitives between the primitive loop and the digestion.  With that, and with
// the density reads of a quartet's digestion issued together, the FP64 build of
// (H2O)32 went from 31.8 to 27.0 ms, the mixed one at 1e-3 from 21.3 to 18.3 ms,
// the B3LYP build of (H2O)64 from 142 to 114 ms.
//
// In run mode (kRuns) a block takes the tiles of one bra pair: the exchange
// contributions to the bra's rows of X are summed in LDS (NA + NB rows of n)
// and added to X once per run, the bra's primitives sit in one LDS slab, and
// its Coulomb block is summed in registers (small blocks) over the run.
// kStaged: run mode with the run's bra rows of the density in LDS after the slab,
// the exchange contractions read there.
// Where a class has too few tiles to fill the GPU, 2^w.lsplit wavefronts share a
// tile in run mode, each taking a part of its primitive quartets, and 2^w.lblocks
// blocks a run (share_tiles): everything after the primitive loop is linear in
// the integrals, so each wavefront digests its own partial sums (one water: 2.39 ->
// 0.54 ms for the build).
template <int LA, int LB, int LC, int LD, typename R, int MODE, class Boys>
__device__ __forceinline__ void fock_quartets(const FockArgs& a, const ClassWork& w, const Boys& boys) {
    constexpr int NE = nrange(LA, LA + LB), NF = nrange(LC, LC + LD);
    constexpr int NACC = NE * NF;
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    constexpr int LT = LA + LB + LC + LD;
    constexpr bool kSliced = HrrSlices<LA, LB, LC, LD>::on;
    constexpr bool RUNS = MODE != kNoRuns, STAGE = MODE == kStaged;
    constexpr bool kKeepJ = RUNS && NA * NB <= 9;   // the run's Coulomb block in registers
    constexpr bool kCentreC = LC + LD > 0;
    using Ft = FockType<R>;
    const R X0 = R(34.98683665524972);  // 2 pi^(5/2), quick_constants_module.f90:55
    const int n = a.n, ns = a.nshell;
    const int lane = threadIdx.x & 63;
    unsigned long long* const Xc = a.X + (long long)(blockIdx.x % a.xcopies) * n * n;
    const int wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned nsurv = 0, nprimq = 0;
    const auto& pp = Ft::prims(a);
    const R* __restrict__ Dp = Ft::density(a);
    const R plim = R(a.prim_limit);
    const int lsplit = RUNS ? w.lsplit : 0;

    // dynamic LDS: in run mode the exchange rows of the run's bra, then that
    // bra's primitive pairs (at most 64; one slab for the block, staged once per
    // run); otherwise one slab per wavefront, staged per tile
    extern __shared__ unsigned long long s_xrows[];
    R* const bra = RUNS ? reinterpret_cast<R*>(s_xrows + (NA + NB) * n)
                        : reinterpret_cast<R*>(s_xrows) + wib * (7 * 64);
    R* const sD = STAGE ? bra + 7 * 64 : nullptr;   // the run's bra rows of D
    const Tile* const tiles = w.steps ? w.steps : w.tiles;
    const bool listed = w.steps != nullptr;

    for (long long run = blockIdx.x;; run += gridDim.x) {
    long long t0, t1, tstep;
    int p = 0;
    if constexpr (RUNS) {
        if ((run >> w.lblocks) >= w.nruns) break;
        const int2 rg = w.runs[run >> w.lblocks];
        tstep = 4ll << w.lblocks;
        t0 = ((long long)rg.x << lsplit) + ((run * 4 + wib) & (tstep - 1)); t1 = (long long)rg.y << lsplit;
        p = w.tiles[rg.x].p;
    } else {
        t0 = (long long)blockIdx.x * 4 + wib; t1 = w.ntiles; tstep = (long long)gridDim.x * 4;
    }
    auto tile_at = [&](long long t) { return t < t1 ? tiles[t >> lsplit] : Tile{0, 0, 0, 0}; };
    auto ket_of = [&](const Tile& tl) { return lane < tl.len ? (listed ? w.list[tl.q0 + lane] : tl.q0 + lane) : 0; };
    Tile T0 = tile_at(t0), T1 = tile_at(t0 + tstep), T2 = tile_at(t0 + 2 * tstep);
    int q0 = ket_of(T0), q1 = ket_of(T1);
    PairRec r0 = a.rec[q0];
    if constexpr (RUNS) {
        for (int k = threadIdx.x; k < (NA + NB) * n; k += blockDim.x) s_xrows[k] = 0ull;
        if (wib == 0) stage_bra(pp, a.pr.prim0[p], a.pr.pstride[p], a.pr.nprim[p], lane, bra);
        if constexpr (STAGE) {
            const unsigned f = a.rec[p].f01;
            const int fa0 = f & 0xffff, fb0 = f >> 16;
            for (int k = threadIdx.x; k < (NA + NB) * n; k += blockDim.x) {
                const int r = k / n, col = k - r * n;
                sD[k] = Dp[(long long)(r < NA ? fa0 + r : fb0 + r - NA) * n + col];
            }
        }
        __syncthreads();
    }
    // a wavefront's share of a tile: bra primitives si, si + 2^lsi, ..., ket
    // primitives sj, sj + 2^(lsplit - lsi), ...; the bra's are split first
    int lsi = 0;
    if constexpr (RUNS)
        while (lsi < lsplit && (1 << lsi) < int((a.rec[p].misc >> 8) & 0x7f)) ++lsi;
    auto share_i = [&](long long t) { return int(t) & ((1 << lsi) - 1); };
    auto share_j = [&](long long t) { return (int(t) & ((1 << lsplit) - 1)) >> lsi; };
    // gathers of a ket's density maxima, centre and first primitive (of the share)
    auto gather = [&](const Tile& tl, const PairRec& r, const unsigned shb, int first) {
        KetGather<R> g;
        const unsigned sC = r.sh & 0xffff, sD_ = r.sh >> 16;
        const double* ca = a.cutmat + (long long)(shb & 0xffff) * ns;
        const double* cb = a.cutmat + (long long)(shb >> 16) * ns;
        g.cd = a.cutmat[(long long)sC * ns + sD_];
        g.ad = ca[sD_]; g.ac = ca[sC]; g.bd = cb[sD_]; g.bc = cb[sC];
        if constexpr (kCentreC) {
            const int at = r.at & 0xffff;
            g.Cx = a.xyz[3 * at]; g.Cy = a.xyz[3 * at + 1]; g.Cz = a.xyz[3 * at + 2];
        }
        // (a lane without a ket holds pair 0, whose primitives lie otherwise)
        const int k = r.prim0 + (lane < tl.len && first < int((r.misc >> 8) & 0x7f) ? first * tl.pad : 0);
        g.z = pp.zeta[k]; g.o = pp.oo2z[k]; g.x = pp.Px[k]; g.y = pp.Py[k]; g.zz = pp.Pz[k];
        g.K = pp.K[k]; g.c = pp.cut[k];
        return g;
    };
    KetGather<R> g0 = gather(T0, r0, a.rec[RUNS ? p : T0.p].sh, share_j(t0));
    long long jac[NA * NB];
#pragma unroll
    for (int k = 0; k < NA * NB; ++k) jac[k] = 0;
    // J on the bra block, in fixed point and so summed exactly across the
    // wavefront (all lanes share the bra pair): one atomic per element
    auto flush_j = [&](const PairRec& rb, int pb) {
        const int fb = rb.f01 >> 16;
#pragma unroll
        for (int k = 0; k < NA * NB; ++k) {
            const long long v = wave_sum_i64(jac[k]);
            jac[k] = 0;
            if (lane == 0 && v != 0) {
                if constexpr (RUNS) atomicAdd(s_xrows + (k / NB) * n + fb + k % NB, (unsigned long long)v);
                else atomicAdd(a.J + rb.jofs + (long long)k * a.pr.pstride[pb], (unsigned long long)v);
            }
        }
    };
    for (long long t = t0; t < t1; t += tstep) {
        if constexpr (!RUNS) p = __builtin_amdgcn_readfirstlane(T0.p);
        const PairRec rb = a.rec[p];
        const PairRec r1 = a.rec[q1];
        const int q2 = ket_of(T2);
        const Tile T3 = tile_at(t + 3 * tstep);
        const int fa = rb.f01 & 0xffff, fb = rb.f01 >> 16;
        const int nbp = (rb.misc >> 8) & 0x7f;
        if constexpr (!RUNS) stage_bra(pp, rb.prim0, a.pr.pstride[p], nbp, lane, bra);   // run mode: staged for the run
        const double dn =
            fmax(fmax(4.0 * a.cutmat[(long long)(rb.sh & 0xffff) * ns + (rb.sh >> 16)], 4.0 * g0.cd),
                 fmax(fmax(g0.ad, g0.ac), fmax(g0.bc, g0.bd)));
        const bool active = lane < T0.len && r0.Y * rb.Y * dn > a.tau;
        R acc[NACC];
#pragma unroll
        for (int k = 0; k < NACC; ++k) acc[k] = R(0);
        const int pks = T0.pad;   // distance of the ket group's consecutive primitives
        if (active) {
            nsurv += (t & ((1 << lsplit) - 1)) == 0;
            const int Mb = a.boys_qshell_order ? LT : int(rb.misc & 15u) + int(r0.misc & 15u);
            const int atA = rb.at & 0xffff;
            const R Ax = R(a.xyz[3 * atA]), Ay = R(a.xyz[3 * atA + 1]), Az = R(a.xyz[3 * atA + 2]);
            const R Cx = kCentreC ? R(g0.Cx) : R(0), Cy = kCentreC ? R(g0.Cy) : R(0), Cz = kCentreC ? R(g0.Cz) : R(0);
            const R dnr = R(dn);
            const int pk0 = r0.prim0, nkp = (r0.misc >> 8) & 0x7f;
            // one primitive quartet: bra primitive i (from the slab) with the ket
            // primitive's data
            auto prims = [&](int i, R zcd, R oo2e, R Qx, R Qy, R Qz, R Kcd, R ccd, R QCx, R QCy, R QCz) {
                if (!((dnr * bra[6 * 64 + i]) * ccd > plim)) return;
                ++nprimq;
                const R zab = bra[i], oo2z = bra[64 + i];
                const R Px = bra[2 * 64 + i], Py = bra[3 * 64 + i], Pz = bra[4 * 64 + i];
                const R rs = rsqrt_nr(zab + zcd);   // 1/sqrt(zeta+eta): reciprocal and root in one
                const R inv = rs * rs;
                const R ROU = zab * (zcd * inv);
                const R Wx = (Px * zab + Qx * zcd) * inv;
                const R Wy = (Py * zab + Qy * zcd) * inv;
                const R Wz = (Pz * zab + Qz * zcd) * inv;
                const R dx = Px - Qx, dy = Py - Qy, dz = Pz - Qz;
                const R T = (dx * dx + dy * dy + dz * dz) * ROU;
                R F[LT + 1];
                const typename Boys::State bs = boys.main(T, F);
                boys.rare(T, Mb, bs, F);
                const R s = X0 * bra[5 * 64 + i] * Kcd * rs;
#pragma unroll
                for (int m = 0; m <= LT; ++m) F[m] *= s;
                ClassOps<LA, LB, LC, LD>::template vrr<R>(F, Px - Ax, Py - Ay, Pz - Az, Wx - Px, Wy - Py, Wz - Pz, QCx,
                                                          QCy, QCz, Wx - Qx, Wy - Qy, Wz - Qz, oo2z, oo2e, R(0.5) * inv,
                                                          zcd * inv, zab * inv, acc);
            };
            // kets outer (vector loads; the next ket primitive is fetched while the
            // current one runs), bra primitives inner, read from the bra slab in LDS
            // (the same address on every lane: broadcast reads)
            R nz = g0.z, no = g0.o, nx = g0.x, ny = g0.y, nzz = g0.zz, nK = g0.K, nc = g0.c;
            const int si = share_i(t), SI = 1 << lsi, SJ = 1 << (lsplit - lsi);
            for (int j = share_j(t); j < nkp; j += SJ) {
                const R zcd = nz, oo2e = no, Qx = nx, Qy = ny, Qz = nzz, Kcd = nK, ccd = nc;
                if (j + SJ < nkp) {
                    const int kn = pk0 + (j + SJ) * pks;
                    nz = pp.zeta[kn]; no = pp.oo2z[kn]; nx = pp.Px[kn]; ny = pp.Py[kn];
                    nzz = pp.Pz[kn]; nK = pp.K[kn]; nc = pp.cut[kn];
                }
                const R QCx = Qx - Cx, QCy = Qy - Cy, QCz = Qz - Cz;
                for (int i = si; i < nbp; i += SI) prims(i, zcd, oo2e, Qx, Qy, Qz, Kcd, ccd, QCx, QCy, QCz);
            }
        }
        const KetGather<R> g1 = gather(T1, r1, RUNS ? rb.sh : a.rec[T1.p].sh, share_j(t + tstep));
        if (active) {
            const int atA = rb.at & 0xffff, atB = rb.at >> 16, atD = r0.at >> 16;
            // digestion: G = (X + X^T)/2 with X accumulating
            //   X[a][b] += 4w D[c][d] I,  X[c][d] += 4w D[a][b] I,
            //   X[a][c] -= h w D[b][d] I, X[a][d] -= h w D[b][c] I,
            //   X[b][c] -= h w D[a][d] I, X[b][d] -= h w D[a][c] I
            // w = 1/((1+[qa==qb])(1+[qc==qd])(1+[p==q])) is the share of the quartet's
            // 8-fold orbit this component set represents.
            const int fc = r0.f01 & 0xffff, fd = r0.f01 >> 16;
            R wgt = R(1);
            if (rb.misc & 16u) wgt *= R(0.5);
            if (r0.misc & 16u) wgt *= R(0.5);
            if (p == q0) wgt *= R(0.5);
            const R jw = R(4) * wgt, kw = -R(a.hybrid) * wgt;
            // exchange: the bra rows of D from LDS (staged per run) or from memory,
            // the sums into the block's LDS rows or straight into X.  No branch
            // between them: the density reads of all of them go out together (a
            // test for zero at each one made every sum wait for its own reads)
            auto put = [&](int r, int grow, int col, R s) {
                const long long iv = Ft::fixed(kw * s);
                if constexpr (RUNS) atomicAdd(s_xrows + r * n + col, (unsigned long long)iv);
                else if (iv != 0) atomicAdd(Xc + (long long)grow * n + col, (unsigned long long)iv);
            };
            R sbc[NB * NC], sbd[NB * ND], scd[NC * ND];
#pragma unroll
            for (int k = 0; k < NB * NC; ++k) sbc[k] = R(0);
#pragma unroll
            for (int k = 0; k < NB * ND; ++k) sbd[k] = R(0);
#pragma unroll
            for (int k = 0; k < NC * ND; ++k) scd[k] = R(0);
            // components [i0, i0 + NS) of A: all at once, or one after another in
            // (dp|pp), whose 162 integrals do not fit in the registers together
            // (private memory 2,128 -> 924 bytes per lane; (H2O)32 3.92 -> 3.27 ms,
            // and with four times the blocks under the scratch bound n-nonane's build
            // 4.34 -> 3.65 ms; (dd|ps) and (dp|ds), 108 integrals, gained nothing or
            // lost: 0.82 -> 1.02 ms)
            auto slice = [&](auto i0_) {
                constexpr int i0 = decltype(i0_)::value, NS = kSliced ? 1 : NA;
                const R* Ds = Dp;
                if constexpr (kSliced) asm volatile("" : "+s"(Ds));   // the reads are not kept from slice to slice
                // element (row, col) of the density; n <= 65535, so the index fits 32 bits
                auto DG = [&](int row, int col) { return Ds[unsigned(row) * unsigned(n) + unsigned(col)]; };
                auto B = [&](int r, int grow, int col) {
                    if constexpr (STAGE) return sD[r * n + col];
                    else return DG(grow, col);
                };
                R out[NS * NB * NC * ND];
                {
                    const R Ax = R(a.xyz[3 * atA]), Ay = R(a.xyz[3 * atA + 1]), Az = R(a.xyz[3 * atA + 2]);
                    const R Bx = R(a.xyz[3 * atB]), By = R(a.xyz[3 * atB + 1]), Bz = R(a.xyz[3 * atB + 2]);
                    R CDx = R(0), CDy = R(0), CDz = R(0);
                    if constexpr (kCentreC) {
                        CDx = R(g0.Cx) - R(a.xyz[3 * atD]);
                        CDy = R(g0.Cy) - R(a.xyz[3 * atD + 1]);
                        CDz = R(g0.Cz) - R(a.xyz[3 * atD + 2]);
                    }
                    if constexpr (kSliced)
                        HrrSlices<LA, LB, LC, LD>::template hrr<i0, R>(acc, Ax - Bx, Ay - By, Az - Bz, CDx, CDy, CDz, out);
                    else
                        ClassOps<LA, LB, LC, LD>::template hrr<R>(acc, Ax - Bx, Ay - By, Az - Bz, CDx, CDy, CDz, out);
                }
#define OUT(is, ib, ic, id) out[(((is)*NB + (ib)) * NC + (ic)) * ND + (id)]
                if (a.hybrid != 0.0) {
                    for (int is = 0; is < NS; ++is)
                        for (int ic = 0; ic < NC; ++ic) {
                            R s = R(0);
                            for (int ib = 0; ib < NB; ++ib)
                                for (int id = 0; id < ND; ++id) s += B(NA + ib, fb + ib, fd + id) * OUT(is, ib, ic, id);
                            put(i0 + is, fa + i0 + is, fc + ic, s);
                        }
                    for (int is = 0; is < NS; ++is)
                        for (int id = 0; id < ND; ++id) {
                            R s = R(0);
                            for (int ib = 0; ib < NB; ++ib)
                                for (int ic = 0; ic < NC; ++ic) s += B(NA + ib, fb + ib, fc + ic) * OUT(is, ib, ic, id);
                            put(i0 + is, fa + i0 + is, fd + id, s);
                        }
                    for (int ib = 0; ib < NB; ++ib)
                        for (int ic = 0; ic < NC; ++ic)
                            for (int is = 0; is < NS; ++is)
                                for (int id = 0; id < ND; ++id)
                                    sbc[ib * NC + ic] += B(i0 + is, fa + i0 + is, fd + id) * OUT(is, ib, ic, id);
                    for (int ib = 0; ib < NB; ++ib)
                        for (int id = 0; id < ND; ++id)
                            for (int is = 0; is < NS; ++is)
                                for (int ic = 0; ic < NC; ++ic)
                                    sbd[ib * ND + id] += B(i0 + is, fa + i0 + is, fc + ic) * OUT(is, ib, ic, id);
                }
                for (int is = 0; is < NS; ++is)
                    for (int ib = 0; ib < NB; ++ib) {
                        R s = R(0);
                        for (int ic = 0; ic < NC; ++ic)
                            for (int id = 0; id < ND; ++id) s += DG(fc + ic, fd + id) * OUT(is, ib, ic, id);
                        jac[(i0 + is) * NB + ib] += Ft::fixed(jw * s);
                    }
                for (int ic = 0; ic < NC; ++ic)
                    for (int id = 0; id < ND; ++id)
                        for (int is = 0; is < NS; ++is)
                            for (int ib = 0; ib < NB; ++ib)
                                scd[ic * ND + id] += DG(fa + i0 + is, fb + ib) * OUT(is, ib, ic, id);
#undef OUT
            };
            for_each_int(std::make_integer_sequence<int, kSliced ? NA : 1>{}, slice);
            if (a.hybrid != 0.0) {
                for (int ib = 0; ib < NB; ++ib)
                    for (int ic = 0; ic < NC; ++ic) put(NA + ib, fb + ib, fc + ic, sbc[ib * NC + ic]);
                for (int ib = 0; ib < NB; ++ib)
                    for (int id = 0; id < ND; ++id) put(NA + ib, fb + ib, fd + id, sbd[ib * ND + id]);
            }
            for (int k = 0; k < NC * ND; ++k) {
                const long long vj = Ft::fixed(jw * scd[k]);
                if (vj != 0) atomicAdd(a.J + r0.jofs + (long long)k * pks, (unsigned long long)vj);
            }
        }
        if constexpr (!kKeepJ) flush_j(rb, p);
        T0 = T1; T1 = T2; T2 = T3;
        q0 = q1; q1 = q2;
        r0 = r1;
        g0 = g1;
    }
    if constexpr (!RUNS) break;
    if constexpr (kKeepJ) flush_j(a.rec[p], p);
    // add the run's rows to X once
    __syncthreads();
    {
        const unsigned f = a.rec[p].f01;
        const int fa0 = f & 0xffff, fb0 = f >> 16;
        for (int k = threadIdx.x; k < (NA + NB) * n; k += blockDim.x) {
            const unsigned long long v = s_xrows[k];
            if (v == 0ull) continue;
            const int r = k / n, col = k - r * n;
            const int grow = r < NA ? fa0 + r : fb0 + (r - NA);
            atomicAdd(Xc + (long long)grow * n + col, v);
        }
    }
    __syncthreads();
    }
    if (nsurv) atomicAdd(a.counters + 0, (unsigned long long)nsurv);
    if (nprimq) atomicAdd(a.counters + 1, (unsigned long long)nprimq);
}

// the two parts of QUICK's fit, with the coefficients in LDS (kernel below)
template <int LT>
struct BoysFit {
    using State = double;   // exp(-T)
    const double* tab;
    __device__ __forceinline__ double main(double T, double* F) const {
        const double E = exp_neg(T);
        boys_fit_main<LT>(T, E, tab, F);
        return E;
    }
    __device__ __forceinline__ void rare(double T, int Mb, double E, double* F) const {
        if (!boys_fit_up(T, Mb)) boys_fit_near0<LT>(T, E, Mb, F);
    }
};

template <int LA, int LB, int LC, int LD, int MODE>
__global__ void __launch_bounds__(256, (Occupancy<LA, LB, LC, LD>::value)) fock_kernel(const FockArgs a, const ClassWork w) {
    __shared__ double s_boys[kBoysFitRegions * kBoysFitTerms];
    for (int k = threadIdx.x; k < kBoysFitRegions * kBoysFitTerms; k += blockDim.x) s_boys[k] = kBoysFit[k];
    __syncthreads();
    fock_quartets<LA, LB, LC, LD, double, MODE>(a, w, BoysFit<LA + LB + LC + LD>{s_boys});
}

// ---------------------------------------------------------------------------
// FP32 path (mixed precision): quartets whose Schwarz bound Y_ij*Y_kl lies
// below the FP32 threshold.  QUICK's Boys fit recurs upward, which is unusable
// in single precision at small T, so this path uses a tabulated Taylor
// expansion of F_LT about the nearest grid point (5 terms, grid 1/8: the
// truncation |d|^5/5! <= 8e-9 relative is below FP32 resolution) and the
// stable downward recursion; beyond T = 36 the asymptotic form and upward
// recursion (the exp(-T) terms are below FP32 resolution there).  The operator
// contributions are promoted to FP64 before the fixed-point accumulation.
//
// The light kernels of the small classes stage the five orders they expand in
// LDS once per block (the per-primitive gather then costs an LDS round trip
// instead of a memory one); where those 5.8 KB would cost resident blocks
// (larger exchange rows, the one-wavefront team kernels) the table is read from
// memory (measured on (H2O)32: (ss|ss) FP32 1.85 -> 1.36 ms with it, (ds|ps)
// 1.28 -> 1.57 ms, dppp gradient 13.5 -> 21.9 ms).
template <int LT>
__device__ __forceinline__ void stage_boys_f32(const float* __restrict__ tab, float* s_tab) {
    for (int i = threadIdx.x; i < kBoysTabRows * kBoysLdsCols; i += blockDim.x) {
        const int k = i / kBoysLdsCols, j = i - k * kBoysLdsCols;
        s_tab[i] = tab[k * kBoysTabM + LT + j];
    }
}

// F_0..F_LT(T) from orders LT..LT+4 of the table: tab points at order LT of
// grid point 0, rows kStride apart (the LDS slice: kBoysLdsCols; the table in
// memory: a.boys_tab + LT and kBoysTabM)
template <int LT, int kStride = kBoysLdsCols>
__device__ __forceinline__ void boys_f32_main(float T, const float* tab, float* F) {
    const int k = __float2int_rn(fminf(T, kBoysTabTmax) * float(kBoysTabPerUnit));
    const float d = float(k) * (1.0f / float(kBoysTabPerUnit)) - T;
    const float* r = tab + k * kStride;
    // F_LT(T) = sum_j F_{LT+j}(T_k) d^j / j!,  d = T_k - T, |d| <= 1/16
    F[LT] = (((r[4] * (d * 0.25f) + r[3]) * (d * (1.0f / 3.0f)) + r[2]) * (d * 0.5f) + r[1]) * d + r[0];
    const float e = __expf(-T);
    const float t2 = T + T;
#pragma unroll
    for (int m = LT - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * (1.0f / float(2 * m + 1));
}
// T >= kBoysTabTmax: sqrt(pi / 4T) by the hardware reciprocal square root
// (no denormal or zero operand here)
template <int LT>
__device__ __forceinline__ void boys_f32_far(float T, float* F) {
    F[0] = 0.88622692545275801f * __builtin_amdgcn_rsqf(T);
    const float h = 0.5f * __builtin_amdgcn_rcpf(T);
#pragma unroll
    for (int m = 1; m <= LT; ++m) F[m] = F[m - 1] * (float(2 * m - 1) * h);
}
template <int LT, int kStride = kBoysLdsCols>
__device__ __forceinline__ void boys_f32(float T, const float* tab, float* F) {
    boys_f32_main<LT, kStride>(T, tab, F);
    if (!(T < kBoysTabTmax)) boys_f32_far<LT>(T, F);
}

// the primitive-pair data, exponents and density in the kernel's precision
template <typename R>
__device__ __forceinline__ const auto& grad_prims(const GradArgs& a) {
    if constexpr (sizeof(R) == 8) return a.pp; else return a.ppf;
}
template <typename R>
__device__ __forceinline__ const R* grad_ea(const GradArgs& a) {
    if constexpr (sizeof(R) == 8) return a.ea; else return a.eaf;
}
template <typename R>
__device__ __forceinline__ const R* grad_eb(const GradArgs& a) {
    if constexpr (sizeof(R) == 8) return a.eb; else return a.ebf;
}
template <typename R>
__device__ __forceinline__ const R* grad_density(const GradArgs& a) {
    if constexpr (sizeof(R) == 8) return a.Dp; else return a.Dpf;
}

// F_0..F_kMaxGradF(T) in FP32 for the gradient's table-driven kernel: the
// expansion of boys_f32 at the highest order the table supports for it (read
// from the table in memory), then downward recursion (stable), so every order
// is valid whatever the class
constexpr int kMaxGradF = 10;
static_assert(kMaxGradF + 4 < kBoysTabM, "Boys table too narrow for the gradient");
__device__ __forceinline__ void boys_f32_all(float T, const float* tab, float* F) {
    boys_f32<kMaxGradF, kBoysTabM>(T, tab + kMaxGradF, F);
}

template <int LA, int LB, int LC, int LD>
struct OccupancyF {
    static constexpr int nacc = nrange(LA, LA + LB) * nrange(LC, LC + LD);
    // six or more exchange rows already hold a run-mode block to three per CU
    // at 800 functions (more functions: fewer): asking for four wavefronts per
    // SIMD only made such kernels spill (measured: ppps 1.34 -> 1.27 ms, dsds
    // 0.44 -> 0.42 ms with three); (dp|pp), with 144 accumulators, spills at two
    // (1.10 -> 0.97 ms with one).  The d-d bras leave run mode above 682 functions,
    // where no rows bound them; (dd|ss) keeps three there and spills 47 registers
    static constexpr int rows = ncart(LA) + ncart(LB);
    static constexpr int value = nacc <= 36 ? (rows >= 6 ? 3 : 4) : (nacc < 144 ? 2 : 1);
};

// the tabulated expansion (kStride: the LDS slice or the table in memory)
template <int LT, int kStride>
struct BoysTab {
    struct State {};
    const float* tab;
    __device__ __forceinline__ State main(float T, float* F) const {
        boys_f32_main<LT, kStride>(T, tab, F);
        return {};
    }
    __device__ __forceinline__ void rare(float T, int, State, float* F) const {
        if (!(T < kBoysTabTmax)) boys_f32_far<LT>(T, F);
    }
};

template <int LA, int LB, int LC, int LD, int MODE>
__global__ void __launch_bounds__(256, (OccupancyF<LA, LB, LC, LD>::value)) fock_kernel_f32(const FockArgs a, const ClassWork w) {
    constexpr int LT = LA + LB + LC + LD;
    constexpr bool kBoysLds = ncart(LA) + ncart(LB) <= 4;   // two or four exchange rows
    __shared__ float s_btab[kBoysLds ? kBoysTabRows * kBoysLdsCols : 1];
    if constexpr (kBoysLds) {
        stage_boys_f32<LT>(a.boys_tab, s_btab);
        __syncthreads();
    }
    constexpr int kStride = kBoysLds ? kBoysLdsCols : kBoysTabM;
    fock_quartets<LA, LB, LC, LD, float, MODE>(a, w, BoysTab<LT, kStride>{kBoysLds ? s_btab : a.boys_tab + LT});
}

// ---------------------------------------------------------------------------
// Schwarz bounds (schwarz.f90:46-548): for every Qshell pair of one pair class,
//   ymax[p]        = max over components of |(ab|ab)| contracted over all
//                    primitive quartets (classcutoff), and
//   pmax[prim i]   = max over components of |[ab|ab]| for the primitive pair i
//                    with itself, weighted by (X0 Xcoeff_i)^2 (classprim).
// The host reduces both over the Qshells of a shell pair and takes sqrt.
template <int LA, int LB>
__global__ void __launch_bounds__(256) schwarz_kernel(const int* __restrict__ pairs, int npairs, const int* __restrict__ pqa,
                                                      const int* __restrict__ pqb, const int* __restrict__ prim0,
                                                      const int* __restrict__ nprim, const DevQshells qs,
                                                      const DevPrims pp, const double* __restrict__ xyz,
                                                      const double* __restrict__ cons,
                                                      double* __restrict__ ymax, double* __restrict__ pmax) {
    constexpr int NE = nrange(LA, LA + LB);
    constexpr int NACC = NE * NE;
    constexpr int NA = ncart(LA), NB = ncart(LB);
    constexpr int NOUT = NA * NB * NA * NB;
    constexpr int LT = 2 * (LA + LB);
    const double X0 = 34.98683665524972;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= npairs) return;
    const int p = pairs[t];
    const int qa = pqa[p], qb = pqb[p];
    const int Mb = 2 * (qs.qfinal[qa] + qs.qfinal[qb]);
    const int atA = qs.atom[qa], atB = qs.atom[qb];
    const double Ax = xyz[3 * atA], Ay = xyz[3 * atA + 1], Az = xyz[3 * atA + 2];
    const double ABx = Ax - xyz[3 * atB], ABy = Ay - xyz[3 * atB + 1], ABz = Az - xyz[3 * atB + 2];
    const int p0 = prim0[p], np = nprim[p];
    double acc[NACC];
    double out[NOUT];
#pragma unroll
    for (int k = 0; k < NACC; ++k) acc[k] = 0.0;
    for (int i = 0; i < np; ++i) {
        const double zab = pp.zeta[p0 + i];
        const double Px = pp.Px[p0 + i], Py = pp.Py[p0 + i], Pz = pp.Pz[p0 + i];
        const double X2 = X0 * pp.K[p0 + i];
        for (int j = 0; j < np; ++j) {
            const double zcd = pp.zeta[p0 + j];
            const double Qx = pp.Px[p0 + j], Qy = pp.Py[p0 + j], Qz = pp.Pz[p0 + j];
            const double ABCD = zab + zcd;
            const double ROU = zab * zcd / ABCD;
            const double Wx = (Px * zab + Qx * zcd) / ABCD, Wy = (Py * zab + Qy * zcd) / ABCD,
                         Wz = (Pz * zab + Qz * zcd) / ABCD;
            const double dx = Px - Qx, dy = Py - Qy, dz = Pz - Qz;
            const double T = (dx * dx + dy * dy + dz * dz) * ROU;
            double F[LT + 1];
            boys_ref<LT>(T, Mb, F);
            const double s = X2 * pp.K[p0 + j] / sqrt(ABCD);
#pragma unroll
            for (int m = 0; m <= LT; ++m) F[m] *= s;
            ClassOps<LA, LB, LA, LB>::template vrr<double>(F, Px - Ax, Py - Ay, Pz - Az, Wx - Px, Wy - Py, Wz - Pz,
                                                           Qx - Ax, Qy - Ay, Qz - Az, Wx - Qx, Wy - Qy, Wz - Qz,
                                                           0.5 / zab, 0.5 / zcd, 0.5 / ABCD, zcd / ABCD, zab / ABCD, acc);
        }
    }
    ClassOps<LA, LB, LA, LB>::template hrr<double>(acc, ABx, ABy, ABz, ABx, ABy, ABz, out);
    // (ab|ab) carries cons(a)^2 cons(b)^2 (hrrwhole's cons product, subs/hrr.f90:295)
    double cab[NA * NB];
    for (int a = 0; a < NA; ++a)
        for (int b = 0; b < NB; ++b) {
            const double ca = cons[qs.f0[qa] + a], cb = cons[qs.f0[qb] + b];
            cab[a * NB + b] = (ca * ca) * (cb * cb);
        }
    double m = 0.0;
    for (int a = 0; a < NA; ++a)
        for (int b = 0; b < NB; ++b) m = fmax(m, fabs(out[((a * NB + b) * NA + a) * NB + b] * cab[a * NB + b]));
    ymax[p] = m;
    // one primitive pair with itself: P = Q, T = 0
    for (int i = 0; i < np; ++i) {
#pragma unroll
        for (int k = 0; k < NACC; ++k) acc[k] = 0.0;
        const double zab = pp.zeta[p0 + i];
        const double Px = pp.Px[p0 + i], Py = pp.Py[p0 + i], Pz = pp.Pz[p0 + i];
        const double ABCD = zab + zab;
        const double Wx = (Px * zab + Px * zab) / ABCD, Wy = (Py * zab + Py * zab) / ABCD,
                     Wz = (Pz * zab + Pz * zab) / ABCD;
        double F[LT + 1];
        boys_ref<LT>(0.0, Mb, F);
        const double x4 = X0 * pp.K[p0 + i];
        const double s = 1.0 / sqrt(ABCD);
#pragma unroll
        for (int k = 0; k <= LT; ++k) F[k] *= s;
        ClassOps<LA, LB, LA, LB>::template vrr<double>(F, Px - Ax, Py - Ay, Pz - Az, Wx - Px, Wy - Py, Wz - Pz,
                                                       Px - Ax, Py - Ay, Pz - Az, Wx - Px, Wy - Py, Wz - Pz,
                                                       0.5 / zab, 0.5 / zab, 0.5 / ABCD, zab / ABCD, zab / ABCD, acc);
#pragma unroll
        for (int k = 0; k < NACC; ++k) acc[k] *= x4 * x4;
        ClassOps<LA, LB, LA, LB>::template hrr<double>(acc, ABx, ABy, ABz, ABx, ABy, ABz, out);
        double mp = 0.0;
        for (int a = 0; a < NA; ++a)
            for (int b = 0; b < NB; ++b) mp = fmax(mp, fabs(out[((a * NB + b) * NA + a) * NB + b] * cab[a * NB + b]));
        pmax[p0 + i] = mp;
    }
}

}  // namespace qk

// qk_grad_light.h -- nuclear gradient with one contracted quartet per lane.
//
// gen_gradw.py generates the arithmetic: the density factors K of a quartet are
// folded through the adjoint horizontal recurrence into weights W_ef once
// (gf_fold), each primitive quartet runs a vertical recurrence raised by one on
// the bra alone and contracts it with W into ten sums (gf_vrr), and the terms
// of dW/d(A-B) and dW/d(C-D) follow from the contracted low-order integrals
// (gf_end).  The form it replaces accumulated four contracted sets raised on
// both sides, recomputing the recurrence in up to four passes, and applied a
// derivative recurrence and a contraction to each set; (pp|pp) held 559 sums
// and 81 density factors there and spilled 4.6 KB a lane, here 126 values in
// chunks.  Measured, whole gradient: n-icosane FP64 100.0 -> 22.9 ms, (H2O)32
// mixed (FP32 below 1e-3) 84.6 -> 22.9 ms; the kernels of (dp|pp) FP64 17.4 ->
// 2.4 ms and of (pp|pp) FP64 12.7 -> 0.83 ms on n-icosane.  What bounds them
// now: FP64 issue at one wavefront per SIMD (30-40% of the SIMD cycles busy)
// in the p and d classes, primitive quartets that fail the primitive screen in
// the s classes.
// Same work tiles, screening, Boys order and weighting as the table-driven
// kernel in qk_grad.hip; the derivative sums of every quartet are converted to
// int64 fixed point (2^-44) and added into a per-block LDS copy of the
// gradient, flushed once per block (or straight into global memory when the
// gradient does not fit in LDS).  The work comes either as tiles (a bra pair
// and up to 64 consecutive kets) or, as the host launches it, compacted by
// compact_kernel to the quartets that pass the screen, packed 64 to a step in
// the tiles' places.
#pragma once
#include "qk_kernels.h"
#include "grad_fold.inc"

#include <utility>

namespace qk {

template <int LA, int LB, int LC, int LD, typename R>
struct GradFold;

#define QK_GRAD_FOLD(la, lb, lc, ld, TAG)              \
    template <>                                        \
    struct GradFold<la, lb, lc, ld, double> {          \
        using type = Fold_##TAG;                       \
    };                                                 \
    template <>                                        \
    struct GradFold<la, lb, lc, ld, float> {           \
        using type = Fold_##TAG##_f;                   \
    };
QK_GRAD_FOLD(0, 0, 0, 0, ssss)
QK_GRAD_FOLD(1, 0, 0, 0, psss)
QK_GRAD_FOLD(1, 0, 1, 0, psps)
QK_GRAD_FOLD(1, 1, 0, 0, ppss)
QK_GRAD_FOLD(2, 0, 0, 0, dsss)
QK_GRAD_FOLD(1, 1, 1, 0, ppps)
QK_GRAD_FOLD(2, 0, 1, 0, dsps)
QK_GRAD_FOLD(2, 1, 0, 0, dpss)
QK_GRAD_FOLD(1, 1, 1, 1, pppp)
QK_GRAD_FOLD(2, 0, 1, 1, dspp)
QK_GRAD_FOLD(2, 0, 2, 0, dsds)
QK_GRAD_FOLD(2, 1, 1, 0, dpps)
QK_GRAD_FOLD(2, 1, 1, 1, dppp)
QK_GRAD_FOLD(2, 1, 2, 0, dpds)
QK_GRAD_FOLD(2, 1, 2, 1, dpdp)
QK_GRAD_FOLD(2, 2, 0, 0, ddss)
QK_GRAD_FOLD(2, 2, 1, 0, ddps)
QK_GRAD_FOLD(2, 2, 1, 1, ddpp)
QK_GRAD_FOLD(2, 2, 2, 0, ddds)
QK_GRAD_FOLD(2, 2, 2, 1, dddp)
#undef QK_GRAD_FOLD

// primitive pairs of the bra for the gradient: the Fock slab's seven fields
// plus the two exponents
template <typename R>
__device__ __forceinline__ void stage_bra_grad(const GradArgs& a, int base, int stride, int n, int lane, R* slab) {
    const auto& P = grad_prims<R>(a);
    const R* ea = grad_ea<R>(a);
    const R* eb = grad_eb<R>(a);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < n) {
        const int k = base + lane * stride;
        slab[lane] = P.zeta[k];
        slab[64 + lane] = P.oo2z[k];
        slab[2 * 64 + lane] = P.Px[k];
        slab[3 * 64 + lane] = P.Py[k];
        slab[4 * 64 + lane] = P.Pz[k];
        slab[5 * 64 + lane] = P.K[k];
        slab[6 * 64 + lane] = P.cut[k];
        slab[7 * 64 + lane] = ea[k];
        slab[8 * 64 + lane] = eb[k];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void gl_add(unsigned long long* lds, unsigned long long* G, bool use_lds, int idx,
                                       double v) {
    const long long iv = __double2ll_rn(v * 0x1p44);
    if (iv == 0) return;
    if (use_lds) atomicAdd(lds + idx, (unsigned long long)iv);
    else atomicAdd(G + idx, (unsigned long long)iv);
}

template <class F, int... K>
__device__ __forceinline__ void for_each_chunk(std::integer_sequence<int, K...>, F&& f) {
    (f(std::integral_constant<int, K>{}), ...);
}

// R = double: QUICK's Boys fit (LDS coefficients); R = float (mixed
// precision, weak quartets): the tabulated Boys expansion of boys_f32, FP32
// arithmetic throughout, the nine sums promoted to FP64 at the accumulate.
template <int LA, int LB, int LC, int LD, typename R>
__global__ void __launch_bounds__(256, (GradFold<LA, LB, LC, LD, R>::type::kWaves)) grad_light_kernel(const GradArgs a, const ClassWork w) {
    using Fd = typename GradFold<LA, LB, LC, LD, R>::type;
    constexpr bool f64 = sizeof(R) == 8;
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    constexpr int LT1 = LA + LB + LC + LD + 1;
    const R X0 = R(34.98683665524972);
    const int n = a.n;
    const int lane = threadIdx.x & 63;
    const long long wave0 = __builtin_amdgcn_readfirstlane(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const long long nwaves = ((long long)gridDim.x * blockDim.x) >> 6;
    unsigned nsurv = 0;
    unsigned long long nprimq = 0;
    extern __shared__ unsigned long long s_grad[];   // 3 x natom when a.lds_grad
    __shared__ double s_boys[f64 ? kBoysFitRegions * kBoysFitTerms : 1];
    __shared__ float s_btab[f64 ? 1 : kBoysTabRows * kBoysLdsCols];
    __shared__ R s_bra[4][9 * 64];
    R* bra = s_bra[threadIdx.x >> 6];
    const bool use_lds = a.lds_grad != 0;
    const auto& PP = grad_prims<R>(a);
    const R* ea = grad_ea<R>(a);
    const R rcut = R(a.cutoff), hyb = R(a.hybrid);
    if constexpr (f64)
        for (int k = threadIdx.x; k < kBoysFitRegions * kBoysFitTerms; k += blockDim.x) s_boys[k] = kBoysFit[k];
    else
        stage_boys_f32<LT1>(a.boys_tab, s_btab);
    if (use_lds)
        for (int k = threadIdx.x; k < 3 * a.natom; k += blockDim.x) s_grad[k] = 0ull;
    __syncthreads();

    // compacted work (w.steps set): the steps written by compact_kernel in the
    // tiles' places, each a bra pair and up to 64 surviving kets in w.list;
    // otherwise tiles of a bra pair and consecutive kets
    const bool compact = w.steps != nullptr;
    // 2^w.lsplit wavefronts share a tile where tiles are few, each taking a part of
    // its primitive quartets: the derivatives are linear in them (one water: 2.28 ->
    // 0.76 ms)
    const int lsplit = w.lsplit;
    for (long long t = wave0; t < w.ntiles << lsplit; t += nwaves) {
        const Tile tl = compact ? w.steps[t >> lsplit] : w.tiles[t >> lsplit];
        const int share = int(t) & ((1 << lsplit) - 1);
        if (tl.len == 0) continue;   // wavefront-uniform: no survivor in this slot
        const int p = __builtin_amdgcn_readfirstlane(tl.p);
        const bool inrange = lane < tl.len;
        const int q = compact ? (inrange ? w.list[tl.q0 + lane] : 0) : tl.q0 + lane;
        const int qa = a.pr.qa[p], qb = a.pr.qb[p];
        const int qc = inrange ? a.pr.qa[q] : 0, qd = inrange ? a.pr.qb[q] : 0;
        const int atA = a.q.atom[qa], atB = a.q.atom[qb], atC = a.q.atom[qc], atD = a.q.atom[qd];
        bool active = false;
        double dn = 0.0;
        if (inrange && !(atA == atB && atA == atC && atA == atD)) {   // one-centre quartets vanish
            const int sA = a.q.shell[qa], sB = a.q.shell[qb], sC = a.q.shell[qc], sD = a.q.shell[qd];
            dn = dn_max(a.cutmat, a.nshell, sA, sB, sC, sD);
            const double ct = a.pr.Y[q] * a.pr.Y[p];
            active = ct > a.cutoff && ct * dn > a.cutoff;
        }
        const int pb0 = a.pr.prim0[p], pbs = a.pr.pstride[p], nbp = a.pr.nprim[p];
        stage_bra_grad<R>(a, pb0, pbs, nbp, lane, bra);
        if (!active) continue;
        nsurv += share == 0;
        // the bra's primitives are split first, then the ket's
        int lsi = 0;
        while (lsi < lsplit && (1 << lsi) < nbp) ++lsi;
        const int si = share & ((1 << lsi) - 1), sj = share >> lsi, SI = 1 << lsi, SJ = 1 << (lsplit - lsi);
        const int Mb = a.q.qfinal[qa] + a.q.qfinal[qb] + a.q.qfinal[qc] + a.q.qfinal[qd] + 2;
        const R Ax = R(a.xyz[3 * atA]), Ay = R(a.xyz[3 * atA + 1]), Az = R(a.xyz[3 * atA + 2]);
        const R Cx = R(a.xyz[3 * atC]), Cy = R(a.xyz[3 * atC + 1]), Cz = R(a.xyz[3 * atC + 2]);
        const R ABx = R(a.xyz[3 * atA] - a.xyz[3 * atB]), ABy = R(a.xyz[3 * atA + 1] - a.xyz[3 * atB + 1]),
                ABz = R(a.xyz[3 * atA + 2] - a.xyz[3 * atB + 2]);
        const R CDx = R(a.xyz[3 * atC] - a.xyz[3 * atD]), CDy = R(a.xyz[3 * atC + 1] - a.xyz[3 * atD + 1]),
                CDz = R(a.xyz[3 * atC + 2] - a.xyz[3 * atD + 2]);
        const int fa = a.q.f0[qa], fb = a.q.f0[qb], fc = a.q.f0[qc], fd = a.q.f0[qd];
        // the share of the quartet's 8-fold orbit this component set represents
        R wq = R(1);
        if (qa == qb) wq *= R(0.5);
        if (qc == qd) wq *= R(0.5);
        if (p == q) wq *= R(0.5);
        // the six density blocks (cons folded into D), scaled so that
        // K = Dab Dcd - (Dac Dbd + Dad Dbc); read again where they are used
        // (the pointer is opaque to the compiler, which would otherwise keep
        // all of them in registers through the primitive loop)
        auto with_density = [&](auto use) {
            const R* D = grad_density<R>(a);
            asm volatile("" : "+s"(D));
            R Dab[NA * NB], Dcd[NC * ND], Dac[NA * NC], Dbd[NB * ND], Dad[NA * ND], Dbc[NB * NC];
            auto block = [&](R* out, int r0, int nr, int c0, int nc, R s) {
#pragma unroll
                for (int i = 0; i < nr; ++i)
#pragma unroll
                    for (int j = 0; j < nc; ++j) out[i * nc + j] = s * D[(long long)(r0 + i) * n + c0 + j];
            };
            block(Dab, fa, NA, fb, NB, R(4) * wq);
            block(Dcd, fc, NC, fd, ND, R(1));
            block(Dac, fa, NA, fc, NC, hyb * wq);
            block(Dbd, fb, NB, fd, ND, R(1));
            block(Dad, fa, NA, fd, ND, hyb * wq);
            block(Dbc, fb, NB, fc, NC, R(1));
            use(Dab, Dcd, Dac, Dbd, Dad, Dbc);
        };
        R g[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) g[k] = R(0);
        const R rdn = R(dn);
        const int pk0 = a.pr.prim0[q], pks = a.pr.pstride[q], nkp = a.pr.nprim[q];
        // one pass over the primitive quartets per chunk of ket functions
        auto pass = [&](auto ktag) {
            constexpr int K = decltype(ktag)::value;
            R W[Fd::kW[K]], S[Fd::kS[K] ? Fd::kS[K] : 1];
#pragma unroll
            for (int k = 0; k < Fd::kW[K]; ++k) W[k] = R(0);
#pragma unroll
            for (int k = 0; k < Fd::kS[K]; ++k) S[k] = R(0);
            with_density([&](const R* Dab, const R* Dcd, const R* Dac, const R* Dbd, const R* Dad, const R* Dbc) {
                Fd::template fold<K, R>(Dab, Dcd, Dac, Dbd, Dad, Dbc, ABx, ABy, ABz, CDx, CDy, CDz, W);
            });
            const int ni = nbp;   // <= 64 primitive pairs per Qshell pair (checked on the host)
            for (int j = sj; j < nkp; j += SJ) {
                const int kj = pk0 + j * pks;
                const R zcd = PP.zeta[kj], oo2e = PP.oo2z[kj];
                const R Qx = PP.Px[kj], Qy = PP.Py[kj], Qz = PP.Pz[kj];
                const R Kcd = PP.K[kj], ccd = PP.cut[kj], ec = ea[kj];
                const R QCx = Qx - Cx, QCy = Qy - Cy, QCz = Qz - Cz;
                const R ge = R(2) * ec * oo2e;                       // gamma / eta
                const R d2 = R(-2) * (zcd - ec);                     // -2 delta
                const R d2x = d2 * CDx, d2y = d2 * CDy, d2z = d2 * CDz;
                for (int i = si; i < ni; i += SI) {
                    if (!((rdn * bra[6 * 64 + i]) * ccd > rcut)) continue;
                    if (K == 0) ++nprimq;
                    const R zab = bra[i], oo2z = bra[64 + i];
                    const R Px = bra[2 * 64 + i], Py = bra[3 * 64 + i], Pz = bra[4 * 64 + i];
                    const R rs = rsqrt_nr(zab + zcd);
                    const R inv = rs * rs;
                    const R roz = zcd * inv, roe = zab * inv;
                    const R ROU = zab * roz;
                    const R Wx = (Px * zab + Qx * zcd) * inv;
                    const R Wy = (Py * zab + Qy * zcd) * inv;
                    const R Wz = (Pz * zab + Qz * zcd) * inv;
                    const R dx = Px - Qx, dy = Py - Qy, dz = Pz - Qz;
                    const R T = (dx * dx + dy * dy + dz * dz) * ROU;
                    R F[LT1 + 1];
                    if constexpr (f64) boys_fit<LT1>(T, Mb, s_boys, F);
                    else boys_f32<LT1>(T, s_btab, F);
                    const R s = X0 * bra[5 * 64 + i] * Kcd * rs;
#pragma unroll
                    for (int m = 0; m <= LT1; ++m) F[m] *= s;
                    R u[10];
#pragma unroll
                    for (int k = 0; k < 10; ++k) u[k] = R(0);
                    Fd::template vrr<K, R>(F, Px - Ax, Py - Ay, Pz - Az, Wx - Px, Wy - Py, Wz - Pz, QCx, QCy, QCz,
                                           Wx - Qx, Wy - Qy, Wz - Qz, oo2z, oo2e, R(0.5) * inv, roz, roe, W, S, u);
                    const R a2 = R(2) * bra[7 * 64 + i], b2 = R(2) * bra[8 * 64 + i], z2 = a2 + b2;
                    const R ex = b2 * ABx, ey = b2 * ABy, ez = b2 * ABz;
                    g[0] += a2 * u[0] - u[4];
                    g[1] += a2 * u[1] - u[5];
                    g[2] += a2 * u[2] - u[6];
                    g[3] += b2 * u[0] + ex * u[3];
                    g[4] += b2 * u[1] + ey * u[3];
                    g[5] += b2 * u[2] + ez * u[3];
                    g[6] += ge * (u[4] + u[7] - z2 * u[0] + (d2x - ex) * u[3]) - u[7];
                    g[7] += ge * (u[5] + u[8] - z2 * u[1] + (d2y - ey) * u[3]) - u[8];
                    g[8] += ge * (u[6] + u[9] - z2 * u[2] + (d2z - ez) * u[3]) - u[9];
                }
            }
            if constexpr (Fd::kS[K] > 0) {
                R tab[3] = {R(0), R(0), R(0)}, tcd[3] = {R(0), R(0), R(0)};
                with_density([&](const R* Dab, const R* Dcd, const R* Dac, const R* Dbd, const R* Dad, const R* Dbc) {
                    Fd::template end<K, R>(Dab, Dcd, Dac, Dbd, Dad, Dbc, ABx, ABy, ABz, CDx, CDy, CDz, S, tab, tcd);
                });
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    g[x] += tab[x];
                    g[3 + x] -= tab[x];
                    g[6 + x] += tcd[x];
                }
            }
        };
        for_each_chunk(std::make_integer_sequence<int, Fd::kChunks>{}, pass);
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const double gA = double(g[x]), gB = double(g[3 + x]), gC = double(g[6 + x]);
            gl_add(s_grad, a.G, use_lds, 3 * atA + x, gA);
            gl_add(s_grad, a.G, use_lds, 3 * atB + x, gB);
            gl_add(s_grad, a.G, use_lds, 3 * atC + x, gC);
            gl_add(s_grad, a.G, use_lds, 3 * atD + x, -(gA + gB + gC));
        }
    }
    if (nsurv) atomicAdd(a.counters + 0, (unsigned long long)nsurv);
    if (nprimq) atomicAdd(a.counters + 1, nprimq);
    if (use_lds) {
        __syncthreads();
        for (int k = threadIdx.x; k < 3 * a.natom; k += blockDim.x)
            if (s_grad[k] != 0ull) atomicAdd(a.G + k, s_grad[k]);
    }
}

}  // namespace qk
